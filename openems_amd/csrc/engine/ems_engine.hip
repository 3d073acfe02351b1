// MI355X (gfx950) EC-FDTD engine: device state, update kernels, extension
// kernels, probes and the C ABI declared in include/ems_hip.h.
//
// Device layout: every field / coefficient array is structure-of-arrays,
// one float32 plane-major block per component, x fastest:
//     a[c * cs + x + Nx * (y + Ny * z)]
// with cs (component stride) rounded up to 64 elements.
//
// Arithmetic follows the reference element update exactly
//     v *= vv;  v += vi * (((a - b) - c) + d)
// (FDTD/engine.cpp:133-168), with separate rounding of every product and sum
// (no contraction: -ffp-contract=off and the pragma below), so results are
// bit-identical to the reference's basic engine on the same operator.
#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>
#include <unordered_map>
#include <thread>
#include <type_traits>
#include <numeric>
#include <vector>

#include "ems_compress.h"
#include "ems_hip.h"

#pragma clang fp contract(off)

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

// a roctx range over a scope (shown by rocprofv3 --marker-trace; free when
// no profiler is attached)
struct TxRange {
    explicit TxRange(const char* m) { roctxRangePushA(m); }
    ~TxRange() { roctxRangePop(); }
    TxRange(const TxRange&) = delete;
    TxRange& operator=(const TxRange&) = delete;
};

#define HIPCHK(expr)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess) return fail(EMS_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr unsigned kBlock = 256;      // threads per block of the stencil kernels (4 wave64)
constexpr unsigned kXCD = 8;          // accelerator complex dies on MI355X
constexpr unsigned kMaxSlabs = 6;     // UPML slabs (Operator_Ext_UPML::Create_UPML creates at most 6)
constexpr size_t kMaxGraphs = 16;     // distinct timestep-chunk graphs kept per engine

struct GridDesc {
    unsigned Nx, Ny, Nz;
    unsigned plane;     // Nx*Ny
    unsigned long long cs;  // component stride
    unsigned zdepth;    // z-sweep depth per block
    unsigned nzc;       // number of z chunks
    unsigned qtiles;    // (x, y) tiles per z chunk
    unsigned tx;        // tile shape: 0 = kBlock consecutive plane positions, else tx x (kBlock/tx) columns
    unsigned ntx;       // tiles along x (2D tiles)
};

// tiles of one z chunk for a tile shape
inline void set_tiles(GridDesc& g, unsigned tx)
{
    g.tx = tx;
    if (tx == 0) {
        g.ntx = 0;
        g.qtiles = (g.plane + kBlock - 1) / kBlock;
    } else {
        const unsigned ty = kBlock / tx;
        g.ntx = (g.Nx + tx - 1) / tx;
        g.qtiles = g.ntx * ((g.Ny + ty - 1) / ty);
    }
    g.nzc = (g.Nz + g.zdepth - 1) / g.zdepth;
}

// (x, y) column of this thread in tile qt, false outside the mesh
__device__ __forceinline__ bool tile_column(const GridDesc& g, unsigned qt, unsigned& x, unsigned& y)
{
    if (g.tx == 0) {
        const unsigned q = qt * kBlock + threadIdx.x;
        y = q / g.Nx;
        x = q - y * g.Nx;
        return q < g.plane;
    }
    const unsigned ty = kBlock / g.tx;
    const unsigned bx = qt % g.ntx, by = qt / g.ntx;
    x = bx * g.tx + threadIdx.x % g.tx;
    y = by * ty + threadIdx.x / g.tx;
    return x < g.Nx && y < g.Ny;
}

// Coefficients of one half step.  Plain layout: SoA arrays cc (vv or ii) and
// cv (vi or iv).  Compressed layout: one uint16 per cell (shared by both half
// steps) into a table of two float4 per entry, {c_x, v_x, c_y, v_y} and
// {c_z, v_z, 0, 0}, one table per half step.
struct CoefArgs {
    const float* cc;
    const float* cv;
    const unsigned short* idx;
    const float4* tab;
    unsigned ntab;                 // float4 entries of tab (2 per unique tuple)
};

// Kernels that stage a small compressed table in LDS first copy it there
// cooperatively (every thread of the workgroup takes part, then a barrier)
// and then read it instead of the global table.
constexpr unsigned kLdsTabBytes = 32768;    // both half steps' tables of the quad sweep

__device__ __forceinline__ void stage_table(float4* dst, const float4* src, unsigned n)
{
    for (unsigned i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
}

// One UPML slab (Operator_Ext_UPML range).  The positions of all slabs are
// numbered consecutively (slab after slab in creation order, x fastest inside
// a slab); every UPML array is [component or coefficient][position].  Along x
// the numbering is padded to whole groups of four cells: it starts at
// xo = x0 rounded down to a multiple of 4 and spans nx (a multiple of 4)
// columns, and every slab starts at a position that is a multiple of 4, so the
// four cells x = 4k .. 4k+3 of a row have four consecutive positions starting
// at a multiple of 4 (16-byte accesses in the quad kernels).  Padding
// positions belong to no cell.
struct SlabTab {
    int x0, x1, y0, y1, z0, z1;    // inclusive mesh ranges
    int xo;                        // x of the numbering's first column (x0 & ~3)
    unsigned nx, ny;               // numbering extents along x (padded) and y
    unsigned long long off;        // number of the slab's first position (a multiple of 4)
};

// UPML of one half step.  Plain UPML: coef[9][npos] = {c0, cfo, cfn} x
// {x, y, z}.  Compressed UPML: pidx[npos] into a table of three float4 per
// entry, {c0_x, c0_y, c0_z, cfo_x}, {cfo_y, cfo_z, cfn_x, cfn_y},
// {cfn_z, 0, 0, 0}.  Flux [3][npos] is read from flux_in and written to
// flux_out (the same buffer when the half step updates in place).  The slab
// table travels in the kernel arguments.
struct PmlArgs {
    int n;                         // number of slabs (0: no UPML)
    unsigned long long npos;
    SlabTab tab[kMaxSlabs];
    const float* coef;
    const unsigned* pidx;
    const float4* ptab;
    const float* flux_in;
    float* flux_out;
};

enum PmlMode { kNoPml = 0, kPmlPlain = 1, kPmlCompressed = 2 };

// Workgroups are dispatched round-robin over the XCDs by linear block id;
// remap so that each XCD owns one contiguous range of tiles (neighbouring
// rows and z-chunks share that XCD's L2).
__device__ __forceinline__ unsigned xcd_tile(unsigned b, unsigned nb)
{
    const unsigned per = nb / kXCD, rem = nb % kXCD;
    const unsigned xcd = b % kXCD, k = b / kXCD;
    return xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
}

// UPML position of cell (x, y, z), or false outside every slab (slabs do not
// overlap; positions fit 32 bits, checked on the host).  The slab is selected
// first and its position computed once.
__device__ __forceinline__ bool pml_at(const PmlArgs& P, int x, int y, int z, unsigned long long& li)
{
    int sel = -1;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        const SlabTab& S = P.tab[s];
        if (s < P.n && x >= S.x0 && x <= S.x1 && y >= S.y0 && y <= S.y1 && z >= S.z0 && z <= S.z1) sel = s;
    }
    int bx = 0, by = 0, bz = 0;
    unsigned nx = 0, ny = 0, off = 0;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        if (sel == s) {
            const SlabTab& S = P.tab[s];
            bx = S.xo; by = S.y0; bz = S.z0;
            nx = S.nx; ny = S.ny; off = (unsigned)S.off;
        }
    }
    li = off + (unsigned)(x - bx) + nx * ((unsigned)(y - by) + ny * (unsigned)(z - bz));
    return sel >= 0;
}

// slabs whose (x, y) range holds column (x, y), one bit per slab
__device__ __forceinline__ unsigned pml_colmask(const PmlArgs& P, int x, int y)
{
    unsigned m = 0;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        const SlabTab& S = P.tab[s];
        if (s < P.n && x >= S.x0 && x <= S.x1 && y >= S.y0 && y <= S.y1) m |= 1u << s;
    }
    return m;
}

// UPML position of (x, y, z) for a column whose slab mask is m; 0 (a valid
// position) when the cell lies in no slab
__device__ __forceinline__ bool pml_at_col(const PmlArgs& P, unsigned m, int x, int y, int z, unsigned& li)
{
    int sel = -1;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        const SlabTab& S = P.tab[s];
        if ((m >> s & 1u) && z >= S.z0 && z <= S.z1) sel = s;
    }
    int bx = 0, by = 0, bz = 0;
    unsigned nx = 0, ny = 0, off = 0;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        if (sel == s) {
            const SlabTab& S = P.tab[s];
            bx = S.xo; by = S.y0; bz = S.z0;
            nx = S.nx; ny = S.ny; off = (unsigned)S.off;
        }
    }
    const unsigned l = off + (unsigned)(x - bx) + nx * ((unsigned)(y - by) + ny * (unsigned)(z - bz));
    li = sel >= 0 ? l : 0u;
    return sel >= 0;
}

// main coefficients of cell p
template <bool CC>
__device__ __forceinline__ void load_coef(const CoefArgs& k, unsigned long long cs, unsigned long long p, unsigned u,
                                          float a[3], float b[3])
{
    if (CC) {
        const float4 t0 = k.tab[2 * u], t1 = k.tab[2 * u + 1];
        a[0] = t0.x; b[0] = t0.y;
        a[1] = t0.z; b[1] = t0.w;
        a[2] = t1.x; b[2] = t1.y;
    } else {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            a[n] = k.cc[n * cs + p];
            b[n] = k.cv[n * cs + p];
        }
    }
}

// Update of the three components of one cell from its old values x0.
//   plain: f = x0*cc + cv*curl;  out = f
//   UPML : f = F*cc + cv*curl;   out = (c0*x0 - cfo*F) + cfn*f;  F <- f
// (F: the UPML flux).  The UPML lanes add exec-masked loads of the flux and
// of their coefficients or table index.  main = false selects the UPML hooks
// alone, out = (c0*x0 - cfo*F) + cfn*F, for a UPML cell the main update
// skips (the caller then stores no flux).
template <int PM>
__device__ __forceinline__ void cell_math(const float x0[3], const float a[3], const float b[3], const float curl[3],
                                          bool pml, const PmlArgs& P, unsigned long long li, bool store_flux,
                                          float out[3], bool main = true)
{
    float k0[3], ko[3], kn[3], fl[3];
    if (PM != kNoPml && pml) {
#pragma unroll
        for (int n = 0; n < 3; ++n) fl[n] = P.flux_in[n * P.npos + li];
    }
    if (PM == kPmlPlain && pml) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            k0[n] = P.coef[n * P.npos + li];
            ko[n] = P.coef[(3 + n) * P.npos + li];
            kn[n] = P.coef[(6 + n) * P.npos + li];
        }
    }
    if (PM == kPmlCompressed && pml) {
        const unsigned u = P.pidx[li];
        const float4 t0 = P.ptab[3 * u], t1 = P.ptab[3 * u + 1], t2 = P.ptab[3 * u + 2];
        k0[0] = t0.x; k0[1] = t0.y; k0[2] = t0.z;
        ko[0] = t0.w; ko[1] = t1.x; ko[2] = t1.y;
        kn[0] = t1.z; kn[1] = t1.w; kn[2] = t2.x;
    }
    float fnew[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const float xin = (PM != kNoPml && pml) ? fl[n] : x0[n];
        float f = xin * a[n];
        f = f + b[n] * curl[n];
        fnew[n] = f;
        if (PM != kNoPml && pml) {
            // a UPML cell the main update skips takes the hooks alone:
            // out = (c0*x0 - cfo*F) + cfn*F (pml_hooks_only)
            const float t = k0[n] * x0[n] - ko[n] * fl[n];
            out[n] = t + kn[n] * (main ? f : fl[n]);
        } else {
            out[n] = f;
        }
    }
    if (PM != kNoPml && pml && store_flux) {
#pragma unroll
        for (int n = 0; n < 3; ++n) P.flux_out[n * P.npos + li] = fnew[n];
    }
}

// UPML hooks alone, for a UPML position the main update skips (the last
// current line of a direction): Engine_Ext_UPML's pre and post hooks run over
// the whole slab (engine_ext_upml.cpp:135-234), so there
//   out = (c0*x0 - cfo*F) + cfn*F,  F unchanged.
template <int PM>
__device__ __forceinline__ void pml_hooks_only(const float x0[3], const PmlArgs& P, unsigned long long li, float out[3])
{
    float k0[3], ko[3], kn[3], fl[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) fl[n] = P.flux_in[n * P.npos + li];
    if (PM == kPmlPlain) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            k0[n] = P.coef[n * P.npos + li];
            ko[n] = P.coef[(3 + n) * P.npos + li];
            kn[n] = P.coef[(6 + n) * P.npos + li];
        }
    } else {
        const unsigned u = P.pidx[li];
        const float4 t0 = P.ptab[3 * u], t1 = P.ptab[3 * u + 1], t2 = P.ptab[3 * u + 2];
        k0[0] = t0.x; k0[1] = t0.y; k0[2] = t0.z;
        ko[0] = t0.w; ko[1] = t1.x; ko[2] = t1.y;
        kn[0] = t1.z; kn[1] = t1.w; kn[2] = t2.x;
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const float t = k0[n] * x0[n] - ko[n] * fl[n];
        out[n] = t + kn[n] * fl[n];
    }
}

// Field accesses of the cell being updated.  It is read and written once per
// launch; on meshes whose fields exceed the last-level cache a non-temporal
// access keeps the caches for the neighbour rows of the other field, which
// adjacent columns and z chunks read again (256^3 PEC: 0.127 -> 0.103 ms per
// half step).  On smaller meshes the fields stay cached from one half step to
// the next, and plain accesses are faster.
template <bool NT>
__device__ __forceinline__ float ld_own(const float* q)
{
    if (NT) return __builtin_nontemporal_load(q);
    return *q;
}

// a cell's coefficient index, read once per half step: non-temporal with
// the own field (256^3 UPML: 0.3361 -> 0.3350 ms per step)
template <bool NT>
__device__ __forceinline__ unsigned cidx(const unsigned short* q)
{
    if (NT) return (unsigned)__builtin_nontemporal_load(q);
    return (unsigned)*q;
}

template <bool NT>
__device__ __forceinline__ void st_own(float* q, float v)
{
    if (NT) __builtin_nontemporal_store(v, q);
    else *q = v;
}

// Excitation entry as the fused step applies it: cell, component, amplitude
// and delay of one Operator_Ext_Excitation list element.
struct ExcEnt {
    unsigned short x, y, z, dir;
    float amp;
    unsigned delay;
};

// sample of the excitation signal at timestep ts for a delay
// (Engine_Ext_Excitation::Apply2Voltages, engine_ext_excitation.cpp:33-61)
__device__ __forceinline__ int exc_sample(int ts, unsigned delay, int period, unsigned length)
{
    const int p = period > 0 ? period : ts + 1;
    int e = ts - (int)delay;
    e *= (e > 0);
    e %= p;
    e *= (e < (int)length);
    return e;
}

struct ExcArgs {
    const unsigned* beg;           // [ntiles + 1] entry ranges per xy tile, each sorted by z
    const ExcEnt* ent;
    const float* sig;
    unsigned length;
    int period;
    const unsigned* tmask;         // k_volt: bit per tile of kBlock columns holding a source (null: every lane looks)
};

// A quad's source entries ordered by plane (list order within a plane):
// [k, e) are the entries not yet applied, nz the plane of entry k (~0u when
// none is left); a sweep that visits planes in increasing order applies each
// plane's entries once and otherwise only compares nz.
struct SrcCursor {
    unsigned k, e, nz;
};

__device__ __forceinline__ SrcCursor src_cursor(const ExcArgs& ex, unsigned b, unsigned e, unsigned z0)
{
    SrcCursor c{b, e, ~0u};
    while (c.k < e && ex.ent[c.k].z < z0) ++c.k;
    if (c.k < e) c.nz = ex.ent[c.k].z;
    return c;
}

// the entries of plane z added to components `mask` of f, in list order
__device__ __forceinline__ void quad_sources_at(const ExcArgs& ex, SrcCursor& c, unsigned x0, unsigned z,
                                                unsigned mask, int ts, float4 f[3])
{
    if (c.nz != z) return;
    unsigned k = c.k;
    for (; k < c.e; ++k) {
        const ExcEnt E = ex.ent[k];
        if (E.z != z) break;
        if (!(mask >> E.dir & 1u)) continue;
        const float sv = E.amp * ex.sig[exc_sample(ts, E.delay, ex.period, ex.length)];
        const unsigned j = (unsigned)E.x - x0;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            if (E.dir != n) continue;
            if (j == 0) f[n].x = f[n].x + sv;
            else if (j == 1) f[n].y = f[n].y + sv;
            else if (j == 2) f[n].z = f[n].z + sv;
            else f[n].w = f[n].w + sv;
        }
    }
    c.k = k;
    c.nz = k < c.e ? ex.ent[k].z : ~0u;
}

// the same for one cell's column (f: its three components)
__device__ __forceinline__ void col_sources_at(const ExcArgs& ex, SrcCursor& c, unsigned z, int ts, float f[3])
{
    if (c.nz != z) return;
    unsigned k = c.k;
    for (; k < c.e; ++k) {
        const ExcEnt E = ex.ent[k];
        if (E.z != z) break;
        const float sv = E.amp * ex.sig[exc_sample(ts, E.delay, ex.period, ex.length)];
        if (E.dir == 0) f[0] = f[0] + sv;
        else if (E.dir == 1) f[1] = f[1] + sv;
        else f[2] = f[2] + sv;
    }
    c.k = k;
    c.nz = k < c.e ? ex.ent[k].z : ~0u;
}

// ---------------------------------------------------------------------------
// voltage half step (Engine::UpdateVoltages, FDTD/engine.cpp:110-168) with the
// UPML pre/post hooks of Engine_Ext_UPML (engine_ext_upml.cpp:52-124) fused in:
//   pre : t = vv_u*V - vvfo*F;  V <- F
//   main: V <- V*vv + vi*curl    (computed on the flux)
//   post: F <- V;  V <- t + vvfn*F
// The lower neighbour at index 0 is the cell itself (shift = bool(pos)).
// Each thread owns one (x, y) column and sweeps g.zdepth planes, carrying the
// z-1 currents in registers.  In place.
// ---------------------------------------------------------------------------
template <int PM, bool CC, bool NT>
__device__ __forceinline__ void volt_tile(const GridDesc& g, unsigned t, float* V, const float* __restrict__ I,
                                          const CoefArgs& k, const PmlArgs& pml, const ExcArgs& ex,
                                          const unsigned* __restrict__ numts)
{
    const unsigned qt = t % g.qtiles, zc = t / g.qtiles;
    unsigned x, y;
    if (!tile_column(g, qt, x, y)) return;
    const unsigned z0 = zc * g.zdepth;
    const unsigned z1 = min(z0 + g.zdepth, g.Nz);
    const unsigned long long cs = g.cs;
    const unsigned xm = x ? 1u : 0u, ym = y ? g.Nx : 0u;
    unsigned long long p = x + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z0;

    const float* __restrict__ Ix = I;
    const float* __restrict__ Iy = I + cs;
    const float* __restrict__ Iz = I + 2 * cs;
    // z-1 values carried in registers along the sweep (self at z = 0)
    const unsigned long long pz = z0 ? p - g.plane : p;
    float Ix_zm = Ix[pz], Iy_zm = Iy[pz];
    // UPML slabs that hold this column (the per-plane test is then along z only)
    const unsigned pcm = PM != kNoPml ? pml_colmask(pml, (int)x, (int)y) : 0u;
    // the column's voltage sources (ordered by plane) where this kernel adds them
    SrcCursor cv{0u, 0u, ~0u};
    int ts = 0;
    if (ex.beg && (!ex.tmask || (ex.tmask[qt >> 5] >> (qt & 31u) & 1u))) {
        cv = src_cursor(ex, ex.beg[x + g.Nx * y], ex.beg[x + g.Nx * y + 1], z0);
        ts = (int)numts[0];
    }

    for (unsigned z = z0; z < z1; ++z, p += g.plane) {
        const float ix = Ix[p], iy = Iy[p], iz = Iz[p];
        const float iz_ym = Iz[p - ym], ix_ym = Ix[p - ym];
        const float iz_xm = Iz[p - xm], iy_xm = Iy[p - xm];
        float curl[3];
        curl[0] = iz - iz_ym - iy + Iy_zm;
        curl[1] = ix - Ix_zm - iz + iz_xm;
        curl[2] = iy - iy_xm - ix + ix_ym;
        Ix_zm = ix;
        Iy_zm = iy;
        float x0[3], a[3], b[3], out[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) x0[n] = ld_own<NT>(&V[n * cs + p]);
        load_coef<CC>(k, cs, p, CC ? cidx<NT>(k.idx + p) : 0u, a, b);
        unsigned li = 0;
        const bool in_pml = PM != kNoPml && pcm && pml_at_col(pml, pcm, (int)x, (int)y, (int)z, li);
        cell_math<PM>(x0, a, b, curl, in_pml, pml, li, true, out);
        col_sources_at(ex, cv, z, ts, out);
#pragma unroll
        for (int n = 0; n < 3; ++n) st_own<NT>(&V[n * cs + p], out[n]);
    }
}

template <int PM, bool CC, bool NT>
__global__ __launch_bounds__(kBlock) void k_volt(const GridDesc g, float* V, const float* __restrict__ I,
                                                 const CoefArgs k, const PmlArgs pml, const ExcArgs ex,
                                                 const unsigned* __restrict__ numts)
{
    volt_tile<PM, CC, NT>(g, xcd_tile(blockIdx.x, gridDim.x), V, I, k, pml, ex, numts);
}

// ---------------------------------------------------------------------------
// current half step (Engine::UpdateCurrents, FDTD/engine.cpp:170-222), same
// UPML fusion with the current flux (engine_ext_upml.cpp:135-234).  Updates
// x < Nx-1, y < Ny-1, z < Nz-1, in place.  Thread (0,0) of tile 0 advances the
// device timestep counter (++numTS of Engine::IterateTS): no kernel of this
// launch reads it, and every later kernel sees the new value.
// ---------------------------------------------------------------------------
template <int PM, bool CC, bool NT>
__device__ __forceinline__ void curr_tile(const GridDesc& g, unsigned t, float* I, const float* __restrict__ V,
                                          const CoefArgs& k, const PmlArgs& pml)
{
    const unsigned qt = t % g.qtiles, zc = t / g.qtiles;
    unsigned x, y;
    if (!tile_column(g, qt, x, y)) return;
    // columns / planes the main update skips only matter for UPML positions
    const bool col_upd = x + 1 < g.Nx && y + 1 < g.Ny;
    if (PM == kNoPml && !col_upd) return;
    const unsigned z0 = zc * g.zdepth;
    const unsigned z1 = min(z0 + g.zdepth, PM == kNoPml ? g.Nz - 1 : g.Nz);
    if (z0 >= z1) return;
    const unsigned long long cs = g.cs;
    // Cells the main update skips (last line of a direction) take the UPML
    // hooks alone, on the same path as the main update: their neighbour
    // loads read the cell itself (valid addresses, values unused), and the
    // result is selected per lane, so a wave holding such a lane does not
    // run a second, serialised branch.
    const unsigned long long dx = col_upd ? 1ull : 0ull, dy = col_upd ? (unsigned long long)g.Nx : 0ull;
    unsigned long long p = x + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z0;

    const float* __restrict__ Vx = V;
    const float* __restrict__ Vy = V + cs;
    const float* __restrict__ Vz = V + 2 * cs;
    // values at z carried from the previous iteration's z+1 loads
    float vx = Vx[p], vy = Vy[p];
    // UPML slabs that hold this column (the per-plane test is then along z only)
    const unsigned pcm = PM != kNoPml ? pml_colmask(pml, (int)x, (int)y) : 0u;

    for (unsigned z = z0; z < z1; ++z, p += g.plane) {
        const bool main = col_upd && z + 1 < g.Nz;
        const unsigned long long pzp = z + 1 < g.Nz ? p + g.plane : p;
        const float vz = Vz[p];
        const float vx_zp = Vx[pzp], vy_zp = Vy[pzp];
        const float vz_yp = Vz[p + dy], vx_yp = Vx[p + dy];
        const float vz_xp = Vz[p + dx], vy_xp = Vy[p + dx];
        float curl[3];
        curl[0] = vz - vz_yp - vy + vy_zp;
        curl[1] = vx - vx_zp - vz + vz_xp;
        curl[2] = vy - vy_xp - vx + vx_yp;
        vx = vx_zp;
        vy = vy_zp;
        float x0[3], a[3], b[3], out[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) x0[n] = ld_own<NT>(&I[n * cs + p]);
        load_coef<CC>(k, cs, p, CC ? cidx<NT>(k.idx + p) : 0u, a, b);
        unsigned li = 0;
        const bool in_pml = PM != kNoPml && pcm && pml_at_col(pml, pcm, (int)x, (int)y, (int)z, li);
        cell_math<PM>(x0, a, b, curl, in_pml, pml, li, main, out, main);
        if (main || in_pml) {
#pragma unroll
            for (int n = 0; n < 3; ++n) st_own<NT>(&I[n * cs + p], out[n]);
        }
    }
}

template <int PM, bool CC, bool NT>
__global__ __launch_bounds__(kBlock) void k_curr(const GridDesc g, float* I, const float* __restrict__ V,
                                                 const CoefArgs k, const PmlArgs pml, unsigned* __restrict__ numts)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(numts, 1u);
    curr_tile<PM, CC, NT>(g, xcd_tile(blockIdx.x, gridDim.x), I, V, k, pml);
}

// ---------------------------------------------------------------------------
// Quad half steps, for meshes with Nx % 4 == 0: each lane owns four
// consecutive x cells (x0 = 4k .. 4k+3) of one row and sweeps z, so every
// field, coefficient and UPML access is 16 bytes per lane (the x-1 / x+1
// neighbour quads are dword-aligned 16-byte loads at p -+ 1).  Per element the
// arithmetic is volt_tile / curr_tile's, in the same order, so the results are
// bit-identical.  A workgroup covers kBlock quads of one z chunk.
// ---------------------------------------------------------------------------
struct alignas(4) F4u {          // four floats at a dword-aligned address
    float v[4];
};

__device__ __forceinline__ float4 ld4u(const float* q)
{
    F4u t;
    __builtin_memcpy(&t, q, 16);
    return make_float4(t.v[0], t.v[1], t.v[2], t.v[3]);
}

typedef float v4f __attribute__((ext_vector_type(4)));

template <bool NT>
__device__ __forceinline__ float4 ld4(const float* q)
{
    if (NT) {
        const v4f t = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(q));
        return make_float4(t.x, t.y, t.z, t.w);
    }
    return *reinterpret_cast<const float4*>(q);
}

template <bool NT>
__device__ __forceinline__ void st4(float* q, float4 v)
{
    if (NT) {
        const v4f t = {v.x, v.y, v.z, v.w};
        __builtin_nontemporal_store(t, reinterpret_cast<v4f*>(q));
    } else {
        *reinterpret_cast<float4*>(q) = v;
    }
}

__device__ __forceinline__ float f4g(const float4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }

__device__ __forceinline__ void f4s(float4& v, int j, float a)
{
    if (j == 0) v.x = a;
    else if (j == 1) v.y = a;
    else if (j == 2) v.z = a;
    else v.w = a;
}

// Boxes of quads a quad half-step launch covers: quads qa .. qa+nq-1 of rows
// ya .. ya+ny-1, planes za .. zb-1, in tiles of kBlock quads (ntiles per z
// chunk of zd planes); `first` is the box's first workgroup.  One box is the whole mesh; a
// UPML mesh splits into the box without UPML cells and the boxes around it.
constexpr int kMaxQBoxes = 8;
struct QBox {
    unsigned qa, nq, ya, ny, za, zb, zd, ntiles, first;   // zd: planes per workgroup
};
// the boxes of one launch in device memory (read with a workgroup-uniform
// index: a by-value array indexed at run time would go to per-lane scratch)
struct QBoxes {
    const QBox* b;
    unsigned n;
};

// quad (x0..x0+3, y) and z range [z0, z1) of lane threadIdx.x in workgroup t;
// false for a lane past its box
__device__ __forceinline__ bool qbox_cell(const QBoxes B, unsigned t, unsigned& x0, unsigned& y, unsigned& z0,
                                          unsigned& z1)
{
    unsigned k = 0;
    for (unsigned i = 1; i < B.n; ++i)
        if (t >= B.b[i].first) k = i;
    const QBox q = B.b[k];
    const unsigned local = t - q.first;
    const unsigned qt = local % q.ntiles, zc = local / q.ntiles;
    const unsigned L = qt * kBlock + threadIdx.x;
    if (L >= q.nq * q.ny) return false;
    const unsigned r = L / q.nq;
    x0 = 4u * (q.qa + (L - r * q.nq));
    y = q.ya + r;
    z0 = q.za + zc * q.zd;
    z1 = min(z0 + q.zd, q.zb);
    return true;
}

// per slab s, bits 4s..4s+3: the elements of quad (x0..x0+3, y) inside the
// slab's x and y ranges
__device__ __forceinline__ unsigned quad_colbits(const PmlArgs& P, int x0, int y)
{
    unsigned m = 0;
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        const SlabTab& S = P.tab[s];
        if (s < P.n && y >= S.y0 && y <= S.y1) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (x0 + j >= S.x0 && x0 + j <= S.x1) m |= 1u << (4 * s + j);
        }
    }
    return m;
}

// UPML part of a quad at plane z.  For every slab holding elements of the
// quad: load the quad's flux (and compressed indices) at the slab's aligned
// position, apply cell_math's UPML formulas to the slab's elements (main: the
// element takes the main update; otherwise the hooks alone), and store the
// flux back (elements outside the slab sit on padding positions and keep
// their values).  in: f[n] = the main update computed on the old values,
// which UPML elements recompute on the flux.
template <int PM, bool STORE_ALL>
__device__ __forceinline__ void quad_pml(const PmlArgs& P, unsigned colbits, int x0, int y, int z, const float4 x0v[3],
                                         const float4 a[3], const float4 b[3], const float4 curl[3], unsigned mainm,
                                         float4 out[3])
{
#pragma unroll
    for (int s = 0; s < (int)kMaxSlabs; ++s) {
        const SlabTab& S = P.tab[s];
        const unsigned bits = (s < P.n && z >= S.z0 && z <= S.z1) ? (colbits >> (4 * s)) & 15u : 0u;
        if (!bits) continue;
        const unsigned li = (unsigned)S.off + (unsigned)(x0 - S.xo) +
                            S.nx * ((unsigned)(y - S.y0) + S.ny * (unsigned)(z - S.z0));
        float4 F[3], Fn[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            F[n] = *reinterpret_cast<const float4*>(P.flux_in + n * P.npos + li);
            Fn[n] = F[n];
        }
        uint4 u4 = make_uint4(0, 0, 0, 0);
        if (PM == kPmlCompressed) u4 = *reinterpret_cast<const uint4*>(P.pidx + li);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (!(bits >> j & 1u)) continue;
            float k0[3], ko[3], kn[3];
            if (PM == kPmlPlain) {
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    k0[n] = P.coef[n * P.npos + li + j];
                    ko[n] = P.coef[(3 + n) * P.npos + li + j];
                    kn[n] = P.coef[(6 + n) * P.npos + li + j];
                }
            } else {
                const unsigned u = j == 0 ? u4.x : j == 1 ? u4.y : j == 2 ? u4.z : u4.w;
                const float4 t0 = P.ptab[3 * u], t1 = P.ptab[3 * u + 1], t2 = P.ptab[3 * u + 2];
                k0[0] = t0.x; k0[1] = t0.y; k0[2] = t0.z;
                ko[0] = t0.w; ko[1] = t1.x; ko[2] = t1.y;
                kn[0] = t1.z; kn[1] = t1.w; kn[2] = t2.x;
            }
            const bool main = mainm >> j & 1u;
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                const float fl = f4g(F[n], j), xo = f4g(x0v[n], j);
                float f = fl * f4g(a[n], j);
                f = f + f4g(b[n], j) * f4g(curl[n], j);
                const float t = k0[n] * xo - ko[n] * fl;
                f4s(out[n], j, t + kn[n] * (main ? f : fl));
                if (STORE_ALL || main) f4s(Fn[n], j, f);
            }
        }
#pragma unroll
        for (int n = 0; n < 3; ++n) *reinterpret_cast<float4*>(P.flux_out + n * P.npos + li) = Fn[n];
    }
}

// main coefficients of the quad at p (p % 4 == 0)
template <bool CC>
__device__ __forceinline__ void quad_coef(const CoefArgs& k, unsigned long long cs, unsigned long long p, float4 a[3],
                                          float4 b[3])
{
    if (CC) {
        const uint2 w = *reinterpret_cast<const uint2*>(k.idx + p);
        const unsigned u[4] = {w.x & 0xFFFFu, w.x >> 16, w.y & 0xFFFFu, w.y >> 16};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 t0 = k.tab[2 * u[j]], t1 = k.tab[2 * u[j] + 1];
            f4s(a[0], j, t0.x); f4s(b[0], j, t0.y);
            f4s(a[1], j, t0.z); f4s(b[1], j, t0.w);
            f4s(a[2], j, t1.x); f4s(b[2], j, t1.y);
        }
    } else {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            a[n] = *reinterpret_cast<const float4*>(k.cc + n * cs + p);
            b[n] = *reinterpret_cast<const float4*>(k.cv + n * cs + p);
        }
    }
}

template <int PM, bool CC, bool NT, bool LT>
__global__ __launch_bounds__(kBlock) void k_volt4(const GridDesc g, const QBoxes boxes, float* V,
                                                  const float* __restrict__ I, const CoefArgs kg, const PmlArgs pml,
                                                  const ExcArgs ex, const unsigned* __restrict__ numts)
{
    extern __shared__ float4 s_tab[];
    CoefArgs k = kg;
    if (LT) {
        stage_table(s_tab, kg.tab, kg.ntab);
        __syncthreads();
        k.tab = s_tab;
    }
    unsigned x0, y, z0, z1;
    if (!qbox_cell(boxes, xcd_tile(blockIdx.x, gridDim.x), x0, y, z0, z1)) return;
    const unsigned long long cs = g.cs;
    unsigned long long p = x0 + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z0;
    const unsigned ym = y ? g.Nx : 0u;
    const unsigned colbits = PM != kNoPml ? quad_colbits(pml, (int)x0, (int)y) : 0u;
    const float* __restrict__ Ix = I;
    const float* __restrict__ Iy = I + cs;
    const float* __restrict__ Iz = I + 2 * cs;
    const unsigned long long pz = z0 ? p - g.plane : p;
    float4 Ix_zm = *reinterpret_cast<const float4*>(Ix + pz), Iy_zm = *reinterpret_cast<const float4*>(Iy + pz);
    // voltage sources added here (per-quad lists ordered by plane) where no
    // hook sits between the update and the excitation; else by the Excite hook
    SrcCursor cv{0u, 0u, ~0u};
    int ts = 0;
    if (ex.beg) {
        const unsigned qi = x0 / 4 + (g.Nx / 4) * y;
        cv = src_cursor(ex, ex.beg[qi], ex.beg[qi + 1], z0);
        ts = (int)numts[0];
    }
    for (unsigned z = z0; z < z1; ++z, p += g.plane) {
        const float4 ix = *reinterpret_cast<const float4*>(Ix + p);
        const float4 iy = *reinterpret_cast<const float4*>(Iy + p);
        const float4 iz = *reinterpret_cast<const float4*>(Iz + p);
        const float4 iz_ym = *reinterpret_cast<const float4*>(Iz + p - ym);
        const float4 ix_ym = *reinterpret_cast<const float4*>(Ix + p - ym);
        // x-1 neighbours: the quad at p-1, or at x0 = 0 the cell itself for element 0
        float4 iz_xm, iy_xm;
        if (x0) {
            iz_xm = ld4u(Iz + p - 1);
            iy_xm = ld4u(Iy + p - 1);
        } else {
            iz_xm = make_float4(iz.x, iz.x, iz.y, iz.z);
            iy_xm = make_float4(iy.x, iy.x, iy.y, iy.z);
        }
        float4 curl[3];
        curl[0].x = iz.x - iz_ym.x - iy.x + Iy_zm.x;
        curl[0].y = iz.y - iz_ym.y - iy.y + Iy_zm.y;
        curl[0].z = iz.z - iz_ym.z - iy.z + Iy_zm.z;
        curl[0].w = iz.w - iz_ym.w - iy.w + Iy_zm.w;
        curl[1].x = ix.x - Ix_zm.x - iz.x + iz_xm.x;
        curl[1].y = ix.y - Ix_zm.y - iz.y + iz_xm.y;
        curl[1].z = ix.z - Ix_zm.z - iz.z + iz_xm.z;
        curl[1].w = ix.w - Ix_zm.w - iz.w + iz_xm.w;
        curl[2].x = iy.x - iy_xm.x - ix.x + ix_ym.x;
        curl[2].y = iy.y - iy_xm.y - ix.y + ix_ym.y;
        curl[2].z = iy.z - iy_xm.z - ix.z + ix_ym.z;
        curl[2].w = iy.w - iy_xm.w - ix.w + ix_ym.w;
        Ix_zm = ix;
        Iy_zm = iy;
        float4 xv[3], a[3], b[3], out[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) xv[n] = ld4<NT>(V + n * cs + p);
        quad_coef<CC>(k, cs, p, a, b);
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            out[n].x = xv[n].x * a[n].x; out[n].x = out[n].x + b[n].x * curl[n].x;
            out[n].y = xv[n].y * a[n].y; out[n].y = out[n].y + b[n].y * curl[n].y;
            out[n].z = xv[n].z * a[n].z; out[n].z = out[n].z + b[n].z * curl[n].z;
            out[n].w = xv[n].w * a[n].w; out[n].w = out[n].w + b[n].w * curl[n].w;
        }
        if (PM != kNoPml) quad_pml<PM, true>(pml, colbits, (int)x0, (int)y, (int)z, xv, a, b, curl, 15u, out);
        quad_sources_at(ex, cv, x0, z, 7u, ts, out);
#pragma unroll
        for (int n = 0; n < 3; ++n) st4<NT>(V + n * cs + p, out[n]);
    }
}

// workgroup `bid` of the half step's `nblk`
template <int PM, bool CC, bool NT, bool LT>
__device__ __forceinline__ void curr4_tile(const GridDesc& g, const QBoxes& boxes, unsigned bid, unsigned nblk, float* I,
                                           const float* __restrict__ V, const CoefArgs& kg, const PmlArgs& pml,
                                           unsigned* __restrict__ numts)
{
    extern __shared__ float4 s_tab[];
    CoefArgs k = kg;
    if (LT) {
        stage_table(s_tab, kg.tab, kg.ntab);
        __syncthreads();
        k.tab = s_tab;
    }
    unsigned x0, y, z0, z1;
    const bool lane = qbox_cell(boxes, xcd_tile(bid, nblk), x0, y, z0, z1);
    // one launch of the half step advances the timestep counter
    if (numts && bid == 0 && threadIdx.x == 0) atomicAdd(numts, 1u);
    if (!lane) return;
    const bool yupd = y + 1 < g.Ny;
    // elements the main update covers along x (x < Nx-1)
    const unsigned xmain = x0 + 4 < g.Nx ? 15u : 7u;
    if (PM == kNoPml && !yupd) return;
    if (PM == kNoPml) z1 = min(z1, g.Nz - 1);
    if (z0 >= z1) return;
    const unsigned long long cs = g.cs;
    const unsigned colbits = PM != kNoPml ? quad_colbits(pml, (int)x0, (int)y) : 0u;
    // neighbours of cells the main update skips read the cell itself
    const unsigned long long dy = yupd ? (unsigned long long)g.Nx : 0ull;
    const bool xlast = x0 + 4 >= g.Nx;
    unsigned long long p = x0 + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z0;
    const float* __restrict__ Vx = V;
    const float* __restrict__ Vy = V + cs;
    const float* __restrict__ Vz = V + 2 * cs;
    float4 vx = *reinterpret_cast<const float4*>(Vx + p), vy = *reinterpret_cast<const float4*>(Vy + p);
    for (unsigned z = z0; z < z1; ++z, p += g.plane) {
        const bool zupd = z + 1 < g.Nz;
        const unsigned mainm = (yupd && zupd) ? xmain : 0u;
        const unsigned long long pzp = zupd ? p + g.plane : p;
        const float4 vz = *reinterpret_cast<const float4*>(Vz + p);
        const float4 vx_zp = *reinterpret_cast<const float4*>(Vx + pzp);
        const float4 vy_zp = *reinterpret_cast<const float4*>(Vy + pzp);
        const float4 vz_yp = *reinterpret_cast<const float4*>(Vz + p + dy);
        const float4 vx_yp = *reinterpret_cast<const float4*>(Vx + p + dy);
        // x+1 neighbours: the quad at p+1, or in the last quad of a row the
        // cell itself for element 3 (its value is not used)
        float4 vz_xp, vy_xp;
        if (!xlast) {
            vz_xp = ld4u(Vz + p + 1);
            vy_xp = ld4u(Vy + p + 1);
        } else {
            vz_xp = make_float4(vz.y, vz.z, vz.w, vz.w);
            vy_xp = make_float4(vy.y, vy.z, vy.w, vy.w);
        }
        float4 curl[3];
        curl[0].x = vz.x - vz_yp.x - vy.x + vy_zp.x;
        curl[0].y = vz.y - vz_yp.y - vy.y + vy_zp.y;
        curl[0].z = vz.z - vz_yp.z - vy.z + vy_zp.z;
        curl[0].w = vz.w - vz_yp.w - vy.w + vy_zp.w;
        curl[1].x = vx.x - vx_zp.x - vz.x + vz_xp.x;
        curl[1].y = vx.y - vx_zp.y - vz.y + vz_xp.y;
        curl[1].z = vx.z - vx_zp.z - vz.z + vz_xp.z;
        curl[1].w = vx.w - vx_zp.w - vz.w + vz_xp.w;
        curl[2].x = vy.x - vy_xp.x - vx.x + vx_yp.x;
        curl[2].y = vy.y - vy_xp.y - vx.y + vx_yp.y;
        curl[2].z = vy.z - vy_xp.z - vx.z + vx_yp.z;
        curl[2].w = vy.w - vy_xp.w - vx.w + vx_yp.w;
        vx = vx_zp;
        vy = vy_zp;
        float4 xv[3], a[3], b[3], out[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) xv[n] = ld4<NT>(I + n * cs + p);
        quad_coef<CC>(k, cs, p, a, b);
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            float4 f;
            f.x = xv[n].x * a[n].x; f.x = f.x + b[n].x * curl[n].x;
            f.y = xv[n].y * a[n].y; f.y = f.y + b[n].y * curl[n].y;
            f.z = xv[n].z * a[n].z; f.z = f.z + b[n].z * curl[n].z;
            f.w = xv[n].w * a[n].w; f.w = f.w + b[n].w * curl[n].w;
            // cells the main update skips keep their values (UPML ones are set below)
            out[n].x = (mainm & 1u) ? f.x : xv[n].x;
            out[n].y = (mainm & 2u) ? f.y : xv[n].y;
            out[n].z = (mainm & 4u) ? f.z : xv[n].z;
            out[n].w = (mainm & 8u) ? f.w : xv[n].w;
        }
        if (PM != kNoPml) quad_pml<PM, false>(pml, colbits, (int)x0, (int)y, (int)z, xv, a, b, curl, mainm, out);
        if (PM != kNoPml || mainm) {
#pragma unroll
            for (int n = 0; n < 3; ++n) st4<NT>(I + n * cs + p, out[n]);
        }
    }
}

template <int PM, bool CC, bool NT, bool LT>
__global__ __launch_bounds__(kBlock) void k_curr4(const GridDesc g, const QBoxes boxes, float* I,
                                                  const float* __restrict__ V, const CoefArgs kg, const PmlArgs pml,
                                                  unsigned* __restrict__ numts)
{
    curr4_tile<PM, CC, NT, LT>(g, boxes, blockIdx.x, gridDim.x, I, V, kg, pml, numts);
}

// ---------------------------------------------------------------------------
// One full timestep in one z-sweep (voltage half step, voltage excitation,
// current half step, current excitation, with UPML fused in both halves):
// the same per-element arithmetic as k_volt / k_curr + the excitation hooks,
// so results are bit-identical to the two-half-step path.
//
// Fields and UPML fluxes are double-buffered: the step reads state n (V0, I0,
// flux_in) and writes state n+1 (V1, I1, flux_out), so workgroups never see
// each other's new values.  A workgroup owns a tile of kTX x kTY (x, y)
// columns and a z chunk; each wave owns 4 rows of 64 columns.  Per plane z it
// computes V^{n+1}(z) for its tile plus a halo (column x0+kTX, row y0+kTY) into
// LDS (the halo values are recomputed, not stored), then I^{n+1}(z-1) from the
// LDS planes z-1 and z.  The first plane of a chunk reads I^n(z0-1) from
// memory; the plane z1 after the chunk is recomputed for I^{n+1}(z1-1).
// Current-side sources must lie inside the updated range (x < Nx-1, ...).
// The last workgroup to finish advances the device timestep counter.
// ---------------------------------------------------------------------------
constexpr unsigned kTX = 64, kTY = 16, kRowsPerWave = kTY / (kBlock / 64);

struct StepArgs {
    GridDesc g;
    unsigned ntx, nty;             // xy tiles
    const float* V0;
    const float* I0;
    float* V1;
    float* I1;
    CoefArgs kV, kI;
    PmlArgs pV, pI;
    ExcArgs eV, eI;
    const unsigned* numts;         // [0] timestep counter (advanced by k_tick or k_curr_again after the step)
};

template <int PM, bool CC>
__device__ __forceinline__ void volt_cell(const StepArgs& a, unsigned x, unsigned y, unsigned z, unsigned long long p,
                                          unsigned u, float ix, float iy, float iz, float ix_zm, float iy_zm,
                                          bool store_flux, int ts, unsigned eb, unsigned ee, float v[3])
{
    const GridDesc& g = a.g;
    const unsigned long long cs = g.cs;
    const unsigned xm = x ? 1u : 0u, ym = y ? g.Nx : 0u;
    const float* __restrict__ I0 = a.I0;
    const float iz_ym = I0[2 * cs + p - ym], ix_ym = I0[p - ym];
    const float iz_xm = I0[2 * cs + p - xm], iy_xm = I0[cs + p - xm];
    float curl[3];
    curl[0] = iz - iz_ym - iy + iy_zm;
    curl[1] = ix - ix_zm - iz + iz_xm;
    curl[2] = iy - iy_xm - ix + ix_ym;
    float x0[3], ca[3], cb[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) x0[n] = a.V0[n * cs + p];
    load_coef<CC>(a.kV, cs, p, u, ca, cb);
    unsigned long long li = 0;
    const bool in_pml = PM != kNoPml && pml_at(a.pV, (int)x, (int)y, (int)z, li);
    cell_math<PM>(x0, ca, cb, curl, in_pml, a.pV, li, store_flux, v);
    // voltage sources of this cell in list order
    for (unsigned e = eb; e < ee; ++e) {
        const ExcEnt E = a.eV.ent[e];
        if (E.z == z && E.x == x && E.y == y) {
            const int s = exc_sample(ts, E.delay, a.eV.period, a.eV.length);
            v[E.dir] = v[E.dir] + E.amp * a.eV.sig[s];
        }
    }
}

// UPML hooks alone at a current cell the main update skips (fused step):
// I^{n+1} from I^n, the flux unchanged (both flux buffers hold it)
template <int PM>
__device__ __forceinline__ void pml_hooks_cell(const StepArgs& a, unsigned x, unsigned y, unsigned z,
                                               unsigned long long p, const float i0[3])
{
    unsigned long long li = 0;
    if (!pml_at(a.pI, (int)x, (int)y, (int)z, li)) return;
    float out[3];
    pml_hooks_only<PM>(i0, a.pI, li, out);
#pragma unroll
    for (int n = 0; n < 3; ++n) a.I1[n * a.g.cs + p] = out[n];
}

template <int PM, bool CC>
__global__ __launch_bounds__(kBlock) void k_step(const StepArgs a)
{
    __shared__ float sV[2][3][kTY + 1][kTX + 1];
    const GridDesc& g = a.g;
    const unsigned long long cs = g.cs;
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned tx = t % a.ntx, ty = (t / a.ntx) % a.nty, zc = t / (a.ntx * a.nty);
    const unsigned tile = tx + a.ntx * ty;
    const unsigned x0 = tx * kTX, y0 = ty * kTY;
    const unsigned z0 = zc * g.zdepth;
    const unsigned z1 = min(z0 + g.zdepth, g.Nz);
    const unsigned zlast = min(z1, g.Nz - 1);
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned x = x0 + lane;
    const int ts = (int)a.numts[0];
    const unsigned evb = a.eV.beg[tile], eve = a.eV.beg[tile + 1];
    const unsigned eib = a.eI.beg[tile], eie = a.eI.beg[tile + 1];
    // halo cells: column x0+kTX (rows 0..kTY) and row y0+kTY (columns 0..kTX-1)
    const bool hcol = x0 + kTX <= g.Nx - 1, hrow = y0 + kTY <= g.Ny - 1;
    const unsigned hi = threadIdx.x;
    const bool h_on_col = hi <= kTY;
    const unsigned hx = h_on_col ? x0 + kTX : x0 + (hi - (kTY + 1));
    const unsigned hy = h_on_col ? y0 + hi : y0 + kTY;
    const bool has_halo = h_on_col ? (hcol && hy < g.Ny) : (hi < kTY + 1 + kTX && hrow && hx < g.Nx);
    const unsigned hr = hy - y0, hc = hx - x0;

    // per row: I^n carried along z (x, y components at z-1) and the own I^n
    // and coefficient index at the previous plane for the current update
    float izm_x[kRowsPerWave], izm_y[kRowsPerWave];
    float iown[kRowsPerWave][3], inew[kRowsPerWave][3];
    unsigned uown[kRowsPerWave], unew[kRowsPerWave];
    const unsigned long long pz0 = z0 ? (unsigned long long)(z0 - 1) * g.plane : 0ull;
#pragma unroll
    for (int r = 0; r < (int)kRowsPerWave; ++r) {
        const unsigned y = y0 + wave * kRowsPerWave + r;
        izm_x[r] = izm_y[r] = 0.0f;
        uown[r] = unew[r] = 0;
        iown[r][0] = iown[r][1] = iown[r][2] = 0.0f;
        inew[r][0] = inew[r][1] = inew[r][2] = 0.0f;
        if (x < g.Nx && y < g.Ny) {
            const unsigned long long p = x + (unsigned long long)g.Nx * y + (z0 ? pz0 : (unsigned long long)z0 * g.plane);
            izm_x[r] = a.I0[p];
            izm_y[r] = a.I0[cs + p];
        }
    }
    float h_izm_x = 0.0f, h_izm_y = 0.0f;
    if (has_halo) {
        const unsigned long long p = hx + (unsigned long long)g.Nx * hy + (z0 ? pz0 : 0ull);
        h_izm_x = a.I0[p];
        h_izm_y = a.I0[cs + p];
    }

    for (unsigned z = z0; z <= zlast; ++z) {
        const unsigned s = z & 1u;
        const unsigned long long zp = (unsigned long long)z * g.plane;
        // -- V^{n+1} at plane z: own rows
#pragma unroll
        for (int r = 0; r < (int)kRowsPerWave; ++r) {
            const unsigned row = wave * kRowsPerWave + r;
            const unsigned y = y0 + row;
            if (x < g.Nx && y < g.Ny) {
                const unsigned long long p = x + (unsigned long long)g.Nx * y + zp;
                const float ix = a.I0[p], iy = a.I0[cs + p], iz = a.I0[2 * cs + p];
                const unsigned u = CC ? a.kV.idx[p] : 0u;
                float v[3];
                volt_cell<PM, CC>(a, x, y, z, p, u, ix, iy, iz, izm_x[r], izm_y[r], z < z1, ts, evb, eve, v);
                izm_x[r] = ix;
                izm_y[r] = iy;
                sV[s][0][row][lane] = v[0];
                sV[s][1][row][lane] = v[1];
                sV[s][2][row][lane] = v[2];
                if (z < z1) {
#pragma unroll
                    for (int n = 0; n < 3; ++n) a.V1[n * cs + p] = v[n];
                }
                // keep I^n and the coefficient index of this cell for I^{n+1}(z)
                inew[r][0] = ix; inew[r][1] = iy; inew[r][2] = iz;
                unew[r] = u;
            }
        }
        // -- halo V^{n+1} at plane z (LDS only)
        if (has_halo) {
            const unsigned long long p = hx + (unsigned long long)g.Nx * hy + zp;
            const float ix = a.I0[p], iy = a.I0[cs + p], iz = a.I0[2 * cs + p];
            const unsigned u = CC ? a.kV.idx[p] : 0u;
            float v[3];
            volt_cell<PM, CC>(a, hx, hy, z, p, u, ix, iy, iz, h_izm_x, h_izm_y, false, ts, evb, eve, v);
            h_izm_x = ix;
            h_izm_y = iy;
            sV[s][0][hr][hc] = v[0];
            sV[s][1][hr][hc] = v[1];
            sV[s][2][hr][hc] = v[2];
        }
        __syncthreads();
        // -- I^{n+1} at plane z-1 from the LDS planes z-1 (slot s^1) and z (slot s)
        if (z > z0) {
            const unsigned zc1 = z - 1;
            const unsigned long long zq = (unsigned long long)zc1 * g.plane;
#pragma unroll
            for (int r = 0; r < (int)kRowsPerWave; ++r) {
                const unsigned row = wave * kRowsPerWave + r;
                const unsigned y = y0 + row;
                if (PM != kNoPml && x < g.Nx && y < g.Ny && !(x + 1 < g.Nx && y + 1 < g.Ny)) {
                    pml_hooks_cell<PM>(a, x, y, zc1, x + (unsigned long long)g.Nx * y + zq, iown[r]);
                } else if (x + 1 < g.Nx && y + 1 < g.Ny) {
                    const unsigned long long p = x + (unsigned long long)g.Nx * y + zq;
                    const unsigned o = s ^ 1u;
                    const float vx = sV[o][0][row][lane], vy = sV[o][1][row][lane], vz = sV[o][2][row][lane];
                    const float vx_zp = sV[s][0][row][lane], vy_zp = sV[s][1][row][lane];
                    const float vz_yp = sV[o][2][row + 1][lane], vx_yp = sV[o][0][row + 1][lane];
                    const float vz_xp = sV[o][2][row][lane + 1], vy_xp = sV[o][1][row][lane + 1];
                    float curl[3];
                    curl[0] = vz - vz_yp - vy + vy_zp;
                    curl[1] = vx - vx_zp - vz + vz_xp;
                    curl[2] = vy - vy_xp - vx + vx_yp;
                    float ca[3], cb[3], out[3];
                    load_coef<CC>(a.kI, cs, p, uown[r], ca, cb);
                    unsigned long long li = 0;
                    const bool in_pml = PM != kNoPml && pml_at(a.pI, (int)x, (int)y, (int)zc1, li);
                    cell_math<PM>(iown[r], ca, cb, curl, in_pml, a.pI, li, true, out);
                    for (unsigned e = eib; e < eie; ++e) {
                        const ExcEnt E = a.eI.ent[e];
                        if (E.z == zc1 && E.x == x && E.y == y) {
                            const int sm = exc_sample(ts, E.delay, a.eI.period, a.eI.length);
                            out[E.dir] = out[E.dir] + E.amp * a.eI.sig[sm];
                        }
                    }
#pragma unroll
                    for (int n = 0; n < 3; ++n) a.I1[n * cs + p] = out[n];
                }
            }
        }
        // I^n and the index of plane z serve the current update at the next plane
#pragma unroll
        for (int r = 0; r < (int)kRowsPerWave; ++r) {
            iown[r][0] = inew[r][0]; iown[r][1] = inew[r][1]; iown[r][2] = inew[r][2];
            uown[r] = unew[r];
        }
        __syncthreads();
    }
    // the last current plane is skipped by the main update: UPML hooks only
    if (PM != kNoPml && z1 == g.Nz) {
        const unsigned long long zq = (unsigned long long)(g.Nz - 1) * g.plane;
#pragma unroll
        for (int r = 0; r < (int)kRowsPerWave; ++r) {
            const unsigned y = y0 + wave * kRowsPerWave + r;
            if (x < g.Nx && y < g.Ny) pml_hooks_cell<PM>(a, x, y, g.Nz - 1, x + (unsigned long long)g.Nx * y + zq, iown[r]);
        }
    }
}

// ---------------------------------------------------------------------------
// Fused single-sweep step without LDS or barriers (k_step2).  The same step as
// k_step (state n in V0, I0 and the flux inputs; state n+1 into V1, I1 and the
// flux outputs), on the two-half-step tiles: a workgroup owns kBlock
// consecutive (x, y) columns and a z chunk, and each thread sweeps its own
// column.  The current update at (x, y, z-1) needs V^{n+1} of its column at
// planes z-1 and z and of the columns (x+1, y) (components z, y) and
// (x, y+1) (components z, x) at plane z-1.  The thread recomputes those four
// neighbour components itself, with the same arithmetic as their owners
// (sources included, flux not stored), and carries plane z-1 in registers,
// so no value crosses threads.  Each plane first issues every load (clamped
// to valid addresses where a value is not needed, so the body has no
// branches before its arithmetic), then computes, then stores.  Sources come
// from per-column lists: the entries of column q are beg[q] .. beg[q+1], in
// list order.
// ---------------------------------------------------------------------------
struct Step2Args {
    GridDesc g;
    CoefArgs kV, kI;
    PmlArgs pV, pI;                // one slab table and index array for both halves
    ExcArgs eV, eI;                // beg: [plane + 1] per-column ranges
    const unsigned* numts;         // [0] timestep counter (advanced by k_tick or k_curr_again after the step)
};

// main coefficients (c, v) of component n at cell p: plain arrays or table
// entry u, whose float2 n is {c_n, v_n}
template <bool CC>
__device__ __forceinline__ float2 coef_n(const CoefArgs& k, unsigned long long cs, unsigned long long p, unsigned u, int n)
{
    if (CC) return reinterpret_cast<const float2*>(k.tab)[4 * u + n];
    return make_float2(k.cc[n * cs + p], k.cv[n * cs + p]);
}

// UPML coefficients (c0, cfo, cfn) of component n at position li: plain
// arrays or the 12 floats of table entry w
template <int PM>
__device__ __forceinline__ void pml_coef_n(const PmlArgs& P, unsigned li, unsigned w, int n, float& k0, float& ko,
                                           float& kn)
{
    if (PM == kPmlPlain) {
        k0 = P.coef[n * P.npos + li];
        ko = P.coef[(3 + n) * P.npos + li];
        kn = P.coef[(6 + n) * P.npos + li];
    } else {
        const float* t = reinterpret_cast<const float*>(P.ptab) + 12 * (unsigned long long)w;
        k0 = t[n];
        ko = t[3 + n];
        kn = t[6 + n];
    }
}

// one component of the update (cell_math for a single component): returns
// the new value, f receives the new flux
template <int PM>
__device__ __forceinline__ float comp_math(float x0, float2 c, float curl, bool pml, float fl, float k0, float ko, float kn,
                                           float& f)
{
    const float xin = (PM != kNoPml && pml) ? fl : x0;
    float g = xin * c.x;
    g = g + c.y * curl;
    f = g;
    if (PM == kNoPml) return g;
    const float t = k0 * x0 - ko * fl;
    const float o = t + kn * g;
    return pml ? o : g;
}

// sources of one column at plane z and component n, added in list order
// (Engine_Ext_Excitation::Apply2Voltages / Apply2Current)
__device__ __forceinline__ float col_sources(const ExcArgs& e, unsigned b, unsigned end, unsigned z, unsigned n, int ts,
                                             float v)
{
    for (unsigned k = b; k < end; ++k) {
        const ExcEnt E = e.ent[k];
        if (E.z == z && E.dir == n) v = v + E.amp * e.sig[exc_sample(ts, E.delay, e.period, e.length)];
    }
    return v;
}

// sources of cell (x, column group) at plane z and component n, from a list
// holding several columns' entries (in list order per cell)
__device__ __forceinline__ float cell_sources(const ExcArgs& e, unsigned b, unsigned end, unsigned x, unsigned z,
                                              unsigned n, int ts, float v)
{
    for (unsigned k = b; k < end; ++k) {
        const ExcEnt E = e.ent[k];
        if (E.x == x && E.z == z && E.dir == n) v = v + E.amp * e.sig[exc_sample(ts, E.delay, e.period, e.length)];
    }
    return v;
}

template <int PM, bool CC>
__global__ __launch_bounds__(kBlock) void k_step2(const Step2Args a, const float* __restrict__ V0,
                                                  const float* __restrict__ I0, float* __restrict__ V1,
                                                  float* __restrict__ I1, const float* __restrict__ fVin,
                                                  float* __restrict__ fVout, const float* __restrict__ fIin,
                                                  float* __restrict__ fIout)
{
    const GridDesc& g = a.g;
    const unsigned long long cs = g.cs;
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned qt = t % g.qtiles, zc = t / g.qtiles;
    unsigned x, y;
    const bool valid = tile_column(g, qt, x, y);
    const int ts = (int)a.numts[0];
    if (valid) {
        const unsigned Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
        const unsigned long long plane = g.plane;
        const unsigned long long npV = a.pV.npos, npI = a.pI.npos;
        const unsigned z0 = zc * g.zdepth;
        const unsigned z1 = min(z0 + g.zdepth, Nz);
        const unsigned zlast = min(z1, Nz - 1);
        const unsigned q = x + Nx * y;
        const bool upd = x + 1 < Nx && y + 1 < Ny;        // the current update runs in this column
        const unsigned long long xm = x ? 1ull : 0ull, ym = y ? (unsigned long long)Nx : 0ull;
        // neighbour columns (the column itself where no current update runs)
        const unsigned long long dr = upd ? 1ull : 0ull, du = upd ? (unsigned long long)Nx : 0ull;
        // source ranges of the own column and of the two neighbour columns
        const unsigned evb = a.eV.beg[q], eve = a.eV.beg[q + 1];
        const unsigned eib = a.eI.beg[q], eie = a.eI.beg[q + 1];
        const unsigned erb = a.eV.beg[q + dr], ere = upd ? a.eV.beg[q + 2] : erb;
        const unsigned eub = a.eV.beg[q + du], eue = upd ? a.eV.beg[q + Nx + 1] : eub;
        unsigned m_own = 0, m_r = 0, m_u = 0;
        if (PM != kNoPml) {
            m_own = pml_colmask(a.pV, (int)x, (int)y);
            if (upd) {
                m_r = pml_colmask(a.pV, (int)x + 1, (int)y);
                m_u = pml_colmask(a.pV, (int)x, (int)y + 1);
            }
        }
        // I^n at z-1 (the cell itself at z = 0): own x, y; (x+1, y) x; (x, y+1) y
        const unsigned long long pzm = z0 ? (unsigned long long)(z0 - 1) * plane + q : (unsigned long long)q;
        float ix_zm = I0[pzm], iy_zm = I0[cs + pzm];
        float ixr_zm = I0[pzm + dr], iyu_zm = I0[cs + pzm + du];
        // plane z-1 carried for the current update: own V^{n+1} and I^n, the
        // neighbour components, the coefficient index, UPML position and index
        float vm0 = 0.0f, vm1 = 0.0f, vm2 = 0.0f, vrz = 0.0f, vry = 0.0f, vuz = 0.0f, vux = 0.0f;
        float im0 = 0.0f, im1 = 0.0f, im2 = 0.0f;
        unsigned um = 0, lim = 0, wm = 0;
        bool pmlm = false;
        unsigned long long pm = q;
        for (unsigned z = z0; z <= zlast; ++z) {
            const unsigned long long p = (unsigned long long)z * plane + q;
            const unsigned long long pr = p + dr, pu = p + du;
            // ---- loads
            const float ix = I0[p], iy = I0[cs + p], iz = I0[2 * cs + p];
            const float iz_ym = I0[2 * cs + p - ym], ix_ym = I0[p - ym];
            const float iz_xm = I0[2 * cs + p - xm], iy_xm = I0[cs + p - xm];
            const float ixr = I0[pr], iyr = I0[cs + pr], izr = I0[2 * cs + pr], ixr_ym = I0[pr - ym];
            const float ixu = I0[pu], iyu = I0[cs + pu], izu = I0[2 * cs + pu], iyu_xm = I0[cs + pu - xm];
            const float v0x = V0[p], v0y = V0[cs + p], v0z = V0[2 * cs + p];
            const float r0z = V0[2 * cs + pr], r0y = V0[cs + pr];
            const float u0z = V0[2 * cs + pu], u0x = V0[pu];
            const unsigned u = CC ? a.kV.idx[p] : 0u;
            const unsigned ur = CC ? a.kV.idx[pr] : 0u;
            const unsigned uu = CC ? a.kV.idx[pu] : 0u;
            const float2 cV0 = coef_n<CC>(a.kV, cs, p, u, 0), cV1 = coef_n<CC>(a.kV, cs, p, u, 1),
                         cV2 = coef_n<CC>(a.kV, cs, p, u, 2);
            const float2 cR2 = coef_n<CC>(a.kV, cs, pr, ur, 2), cR1 = coef_n<CC>(a.kV, cs, pr, ur, 1);
            const float2 cU2 = coef_n<CC>(a.kV, cs, pu, uu, 2), cU0 = coef_n<CC>(a.kV, cs, pu, uu, 0);
            const float2 cI0 = coef_n<CC>(a.kI, cs, pm, um, 0), cI1 = coef_n<CC>(a.kI, cs, pm, um, 1),
                         cI2 = coef_n<CC>(a.kI, cs, pm, um, 2);
            unsigned li = 0, lr = 0, lu = 0, w = 0;
            bool pml = false, pmr = false, pmu = false;
            float fl[3] = {0.0f, 0.0f, 0.0f}, k0[3] = {0.0f, 0.0f, 0.0f}, ko[3] = {0.0f, 0.0f, 0.0f},
                  kn[3] = {0.0f, 0.0f, 0.0f};
            float flr2 = 0.0f, flr1 = 0.0f, flu2 = 0.0f, flu0 = 0.0f;
            float kr[2][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}}, ku[2][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            float flI[3] = {0.0f, 0.0f, 0.0f}, kI0[3] = {0.0f, 0.0f, 0.0f}, kIo[3] = {0.0f, 0.0f, 0.0f},
                  kIn[3] = {0.0f, 0.0f, 0.0f};
            if (PM != kNoPml) {
                pml = pml_at_col(a.pV, m_own, (int)x, (int)y, (int)z, li);
                pmr = pml_at_col(a.pV, m_r, (int)x + 1, (int)y, (int)z, lr);
                pmu = pml_at_col(a.pV, m_u, (int)x, (int)y + 1, (int)z, lu);
                w = PM == kPmlCompressed ? a.pV.pidx[li] : 0u;
                const unsigned wr = PM == kPmlCompressed ? a.pV.pidx[lr] : 0u;
                const unsigned wu = PM == kPmlCompressed ? a.pV.pidx[lu] : 0u;
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    fl[n] = fVin[n * npV + li];
                    pml_coef_n<PM>(a.pV, li, w, n, k0[n], ko[n], kn[n]);
                    flI[n] = fIin[n * npI + lim];
                    pml_coef_n<PM>(a.pI, lim, wm, n, kI0[n], kIo[n], kIn[n]);
                }
                flr2 = fVin[2 * npV + lr];
                flr1 = fVin[npV + lr];
                pml_coef_n<PM>(a.pV, lr, wr, 2, kr[0][0], kr[0][1], kr[0][2]);
                pml_coef_n<PM>(a.pV, lr, wr, 1, kr[1][0], kr[1][1], kr[1][2]);
                flu2 = fVin[2 * npV + lu];
                flu0 = fVin[lu];
                pml_coef_n<PM>(a.pV, lu, wu, 2, ku[0][0], ku[0][1], ku[0][2]);
                pml_coef_n<PM>(a.pV, lu, wu, 0, ku[1][0], ku[1][1], ku[1][2]);
            }
            // ---- own V^{n+1}(x, y, z)
            float v[3], fv[3];
            {
                const float c0 = iz - iz_ym - iy + iy_zm;
                const float c1 = ix - ix_zm - iz + iz_xm;
                const float c2 = iy - iy_xm - ix + ix_ym;
                v[0] = comp_math<PM>(v0x, cV0, c0, pml, fl[0], k0[0], ko[0], kn[0], fv[0]);
                v[1] = comp_math<PM>(v0y, cV1, c1, pml, fl[1], k0[1], ko[1], kn[1], fv[1]);
                v[2] = comp_math<PM>(v0z, cV2, c2, pml, fl[2], k0[2], ko[2], kn[2], fv[2]);
            }
            // ---- neighbour components: (x+1, y) z and y, (x, y+1) z and x
            float nrz, nry, nuz, nux, dummy;
            {
                const float c2r = iyr - iy - ixr + ixr_ym;
                const float c1r = ixr - ixr_zm - izr + iz;
                nrz = comp_math<PM>(r0z, cR2, c2r, pmr, flr2, kr[0][0], kr[0][1], kr[0][2], dummy);
                nry = comp_math<PM>(r0y, cR1, c1r, pmr, flr1, kr[1][0], kr[1][1], kr[1][2], dummy);
                const float c2u = iyu - iyu_xm - ixu + ix;
                const float c0u = izu - iz - iyu + iyu_zm;
                nuz = comp_math<PM>(u0z, cU2, c2u, pmu, flu2, ku[0][0], ku[0][1], ku[0][2], dummy);
                nux = comp_math<PM>(u0x, cU0, c0u, pmu, flu0, ku[1][0], ku[1][1], ku[1][2], dummy);
            }
            // ---- voltage sources
            if (evb != eve) {
#pragma unroll
                for (int n = 0; n < 3; ++n) v[n] = col_sources(a.eV, evb, eve, z, n, ts, v[n]);
            }
            if (erb != ere) {
                nrz = col_sources(a.eV, erb, ere, z, 2, ts, nrz);
                nry = col_sources(a.eV, erb, ere, z, 1, ts, nry);
            }
            if (eub != eue) {
                nuz = col_sources(a.eV, eub, eue, z, 2, ts, nuz);
                nux = col_sources(a.eV, eub, eue, z, 0, ts, nux);
            }
            // ---- I^{n+1}(x, y, z-1): main update, or the UPML hooks alone in
            // a column the main update skips
            float io[3], fi[3];
            {
                const float c0 = vm2 - vuz - vm1 + v[1];
                const float c1 = vm0 - v[0] - vm2 + vrz;
                const float c2 = vm1 - vry - vm0 + vux;
                const float im[3] = {im0, im1, im2};
                io[0] = comp_math<PM>(im[0], cI0, c0, pmlm, flI[0], kI0[0], kIo[0], kIn[0], fi[0]);
                io[1] = comp_math<PM>(im[1], cI1, c1, pmlm, flI[1], kI0[1], kIo[1], kIn[1], fi[1]);
                io[2] = comp_math<PM>(im[2], cI2, c2, pmlm, flI[2], kI0[2], kIo[2], kIn[2], fi[2]);
                if (PM != kNoPml && !upd) {
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        const float tt = kI0[n] * im[n] - kIo[n] * flI[n];
                        io[n] = tt + kIn[n] * flI[n];
                    }
                }
            }
            const bool wI = z > z0 && (upd || (PM != kNoPml && pmlm));
            if (z > z0 && upd && eib != eie) {
#pragma unroll
                for (int n = 0; n < 3; ++n) io[n] = col_sources(a.eI, eib, eie, z - 1, n, ts, io[n]);
            }
            // ---- stores
            if (z < z1) {
                V1[p] = v[0];
                V1[cs + p] = v[1];
                V1[2 * cs + p] = v[2];
                if (PM != kNoPml && pml) {
                    fVout[li] = fv[0];
                    fVout[npV + li] = fv[1];
                    fVout[2 * npV + li] = fv[2];
                }
            }
            if (wI) {
                I1[pm] = io[0];
                I1[cs + pm] = io[1];
                I1[2 * cs + pm] = io[2];
                if (PM != kNoPml && pmlm && upd) {
                    fIout[lim] = fi[0];
                    fIout[npI + lim] = fi[1];
                    fIout[2 * npI + lim] = fi[2];
                }
            }
            // ---- carry plane z
            vm0 = v[0]; vm1 = v[1]; vm2 = v[2];
            vrz = nrz; vry = nry; vuz = nuz; vux = nux;
            im0 = ix; im1 = iy; im2 = iz;
            ix_zm = ix; iy_zm = iy;
            ixr_zm = ixr; iyu_zm = iyu;
            um = u; lim = li; wm = w; pmlm = pml;
            pm = p;
        }
        // the last current plane is skipped by the main update: UPML hooks only
        if (PM != kNoPml && z1 == Nz && pmlm) {
            const float im[3] = {im0, im1, im2};
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                float c0, co, cn;
                pml_coef_n<PM>(a.pI, lim, wm, n, c0, co, cn);
                const float fl = fIin[n * npI + lim];
                const float tt = c0 * im[n] - co * fl;
                I1[n * cs + pm] = tt + cn * fl;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Quad column sweep: one full timestep per launch, four x cells per lane
// (16-byte accesses), over a box of cells without UPML (k_step2's scheme with
// quads).  Each lane owns the quad x0 .. x0+3 of row y and sweeps a z chunk;
// per plane z it loads state n once and computes
//   * V^{n+1}(x0..x0+3, y, z), stored;
//   * V^{n+1} z and x components of the quad of row y+1 and z and y
//     components of the cell (x0+4, y): the neighbours its current update
//     reads, recomputed (not stored) with their owners' arithmetic, sources
//     included;
//   * I^{n+1}(x0..x0+3, y, z-1) from those, stored.
// The box is [4*qa, 4*(qa+nq)) x [ya, ya+ny) x [za, zb); voltages are stored
// on all of it, currents where x + 1 < xb, y + 1 < yb and z + 1 < zb (the
// rest of the box's current update, and every cell outside the box, belongs
// to another pass or to no update at all).  Per element the arithmetic is
// k_step2's (and so k_volt / k_curr's): results are bit-identical.
// ---------------------------------------------------------------------------
// A Mur face on x = 0 (neighbour line 1) or x = Nx-1 (neighbour Nx-2) whose
// pre and post hooks k_step4t runs (its points are numbered z * Ny + y)
struct MurFold {
    const float* cP;               // coefficients of the y and z components
    const float* cPP;
    float* mP;                     // the hooks' values, read by the MurApply hook
    float* mPP;
    unsigned start_ts;
    unsigned on;
};

struct Step4Args {
    GridDesc g;
    CoefArgs kV, kI;
    ExcArgs eV, eI;                // beg: [plane + 1] per-column ranges in list order
    const unsigned* numts;
    unsigned qa, nq, ya, ny, za, zb, xb, yb;
    unsigned zdepth, ntiles;       // planes per chunk; tiles of kBlock quads over nq * ny
    unsigned ntq;                  // k_step4t: tiles of 64 quads along x (ntiles = ntq x row tiles)
    MurFold mf[2];                 // k_step4t: the x = 0 and x = Nx-1 Mur faces
};

// coefficient pair (c, v) of component n of the quad at p (table entries u[])
template <bool CC>
__device__ __forceinline__ void quad_coef_n(const CoefArgs& k, unsigned long long cs, unsigned long long p,
                                            const unsigned u[4], int n, float4& c, float4& v)
{
    if (CC) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float2 t = reinterpret_cast<const float2*>(k.tab)[4 * u[j] + n];
            f4s(c, j, t.x);
            f4s(v, j, t.y);
        }
    } else {
        c = *reinterpret_cast<const float4*>(k.cc + n * cs + p);
        v = *reinterpret_cast<const float4*>(k.cv + n * cs + p);
    }
}

__device__ __forceinline__ void quad_idx(const unsigned short* idx, unsigned long long p, unsigned u[4])
{
    const uint2 w = *reinterpret_cast<const uint2*>(idx + p);
    u[0] = w.x & 0xFFFFu;
    u[1] = w.x >> 16;
    u[2] = w.y & 0xFFFFu;
    u[3] = w.y >> 16;
}

__device__ __forceinline__ float4 quad_math(float4 x0, float4 c, float4 v, float4 curl)
{
    float4 o;
    o.x = x0.x * c.x; o.x = o.x + v.x * curl.x;
    o.y = x0.y * c.y; o.y = o.y + v.y * curl.y;
    o.z = x0.z * c.z; o.z = o.z + v.z * curl.z;
    o.w = x0.w * c.w; o.w = o.w + v.w * curl.w;
    return o;
}

// a - b - c + d per element, in that order
__device__ __forceinline__ float4 quad_curl(float4 a, float4 b, float4 c, float4 d)
{
    float4 o;
    o.x = a.x - b.x - c.x + d.x;
    o.y = a.y - b.y - c.y + d.y;
    o.z = a.z - b.z - c.z + d.z;
    o.w = a.w - b.w - c.w + d.w;
    return o;
}

// the sources of columns x0 .. x0+3 (entries [b, e), list order) at plane z
// added to components `mask` (bit n: component n) of f
__device__ __forceinline__ void quad_sources(const ExcArgs& ex, unsigned b, unsigned e, unsigned x0, unsigned z,
                                             unsigned mask, int ts, float4 f[3])
{
    for (unsigned k = b; k < e; ++k) {
        const ExcEnt E = ex.ent[k];
        if (E.z != z || !(mask >> E.dir & 1u)) continue;
        const float sv = E.amp * ex.sig[exc_sample(ts, E.delay, ex.period, ex.length)];
        const unsigned j = (unsigned)E.x - x0;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            if (E.dir != n) continue;
            if (j == 0) f[n].x = f[n].x + sv;
            else if (j == 1) f[n].y = f[n].y + sv;
            else if (j == 2) f[n].z = f[n].z + sv;
            else f[n].w = f[n].w + sv;
        }
    }
}

template <bool CC, bool NT, bool LT>
__global__ __launch_bounds__(kBlock) void k_step4(const Step4Args ag, const float* __restrict__ V0,
                                                  const float* __restrict__ I0, float* __restrict__ V1,
                                                  float* __restrict__ I1)
{
    extern __shared__ float4 s_tab[];
    Step4Args a = ag;
    if (LT) {
        stage_table(s_tab, ag.kV.tab, ag.kV.ntab);
        stage_table(s_tab + ag.kV.ntab, ag.kI.tab, ag.kI.ntab);
        __syncthreads();
        a.kV.tab = s_tab;
        a.kI.tab = s_tab + ag.kV.ntab;
    }
    const GridDesc& g = a.g;
    const unsigned long long cs = g.cs;
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned qt = t % a.ntiles, zc = t / a.ntiles;
    const unsigned L = qt * kBlock + threadIdx.x;
    if (L >= a.nq * a.ny) return;
    const unsigned r = L / a.nq;
    const unsigned x0 = 4u * (a.qa + (L - r * a.nq)), y = a.ya + r;
    const int ts = (int)a.numts[0];
    const unsigned Nx = g.Nx;
    const unsigned long long plane = g.plane;
    const unsigned z0 = a.za + zc * a.zdepth;
    const unsigned z1 = min(z0 + a.zdepth, a.zb);
    // the plane after the chunk is recomputed for the currents of its last plane
    const unsigned zlast = z1 < a.zb ? z1 : z1 - 1;
    const unsigned q = x0 + Nx * y;
    const bool yupd = y + 1 < a.yb;                    // the row's current update runs here
    const bool xr = x0 + 4 < a.xb;                     // element 3's current update runs here
    const unsigned imask = !yupd ? 0u : xr ? 15u : (x0 + 3 < a.xb ? 7u : x0 + 2 < a.xb ? 3u : x0 + 1 < a.xb ? 1u : 0u);
    const unsigned long long ym = y ? (unsigned long long)Nx : 0ull;
    // neighbours read by the current update (the cell itself where none runs)
    const unsigned long long du = yupd ? (unsigned long long)Nx : 0ull, dr = xr ? 4ull : 0ull;
    const unsigned evb = a.eV.beg[q], eve = a.eV.beg[q + 4];
    const unsigned eib = a.eI.beg[q], eie = a.eI.beg[q + 4];
    const unsigned eub = a.eV.beg[q + du], eue = yupd ? a.eV.beg[q + du + 4] : eub;
    // cell x0+4: the next quad's list (ordered by plane), entries of x0+4 only
    const unsigned erb = a.eV.beg[q + dr], ere = xr ? a.eV.beg[q + dr + 4] : erb;
    // V^{n+1} of plane z-1 carried for the current update: the own quad, the
    // z and x components of row y+1, the z and y components of (x0+4, y)
    float4 vm[3] = {}, vu2m = {}, vu0m = {};
    float vr2m = 0.0f, vr1m = 0.0f;
    for (unsigned z = z0; z <= zlast; ++z) {
        const unsigned long long p = (unsigned long long)z * plane + q;
        // I^n at z-1 (the cell itself at z = 0); read again where needed
        const unsigned long long pz = z ? p - plane : p;
        // ---- own V^{n+1}(x0..x0+3, y, z)
        const float4 ix = *reinterpret_cast<const float4*>(I0 + p);
        const float4 iy = *reinterpret_cast<const float4*>(I0 + cs + p);
        const float4 iz = *reinterpret_cast<const float4*>(I0 + 2 * cs + p);
        float4 v[3];
        unsigned u[4] = {0u, 0u, 0u, 0u};
        {
            const float4 iz_ym = *reinterpret_cast<const float4*>(I0 + 2 * cs + p - ym);
            const float4 ix_ym = *reinterpret_cast<const float4*>(I0 + p - ym);
            const float4 ix_m = *reinterpret_cast<const float4*>(I0 + pz);
            const float4 iy_m = *reinterpret_cast<const float4*>(I0 + cs + pz);
            float4 iz_xm, iy_xm;
            if (x0) {
                iz_xm = ld4u(I0 + 2 * cs + p - 1);
                iy_xm = ld4u(I0 + cs + p - 1);
            } else {
                iz_xm = make_float4(iz.x, iz.x, iz.y, iz.z);
                iy_xm = make_float4(iy.x, iy.x, iy.y, iy.z);
            }
            float4 v0[3];
            v0[0] = ld4<NT>(V0 + p);
            v0[1] = ld4<NT>(V0 + cs + p);
            v0[2] = ld4<NT>(V0 + 2 * cs + p);
            if (CC) quad_idx(a.kV.idx, p, u);
            float4 c, w;
            quad_coef_n<CC>(a.kV, cs, p, u, 0, c, w);
            v[0] = quad_math(v0[0], c, w, quad_curl(iz, iz_ym, iy, iy_m));
            quad_coef_n<CC>(a.kV, cs, p, u, 1, c, w);
            v[1] = quad_math(v0[1], c, w, quad_curl(ix, ix_m, iz, iz_xm));
            quad_coef_n<CC>(a.kV, cs, p, u, 2, c, w);
            v[2] = quad_math(v0[2], c, w, quad_curl(iy, iy_xm, ix, ix_ym));
            if (evb != eve) quad_sources(a.eV, evb, eve, x0, z, 7u, ts, v);
        }
        if (z < z1) {
#pragma unroll
            for (int n = 0; n < 3; ++n) st4<NT>(V1 + n * cs + p, v[n]);
        }
        // ---- I^{n+1}(x0..x0+3, y, z-1) from the carried plane and v
        if (z > z0 && z < a.zb && imask) {
            const unsigned long long pm = pz;
            unsigned um[4] = {0u, 0u, 0u, 0u};
            if (CC) quad_idx(a.kI.idx, pm, um);
            float4 io[3];
            const float4 vzr = make_float4(vm[2].y, vm[2].z, vm[2].w, vr2m);
            const float4 vyr = make_float4(vm[1].y, vm[1].z, vm[1].w, vr1m);
            float4 c, w;
            quad_coef_n<CC>(a.kI, cs, pm, um, 0, c, w);
            io[0] = quad_math(*reinterpret_cast<const float4*>(I0 + pm), c, w, quad_curl(vm[2], vu2m, vm[1], v[1]));
            quad_coef_n<CC>(a.kI, cs, pm, um, 1, c, w);
            io[1] = quad_math(*reinterpret_cast<const float4*>(I0 + cs + pm), c, w, quad_curl(vm[0], v[0], vm[2], vzr));
            quad_coef_n<CC>(a.kI, cs, pm, um, 2, c, w);
            io[2] = quad_math(*reinterpret_cast<const float4*>(I0 + 2 * cs + pm), c, w,
                              quad_curl(vm[1], vyr, vm[0], vu0m));
            if (eib != eie) quad_sources(a.eI, eib, eie, x0, z - 1, 7u, ts, io);
            if (imask == 15u) {
#pragma unroll
                for (int n = 0; n < 3; ++n) st4<NT>(I1 + n * cs + pm, io[n]);
            } else {
#pragma unroll
                for (int n = 0; n < 3; ++n)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (imask >> j & 1u) I1[n * cs + pm + j] = f4g(io[n], j);
            }
        }
        vm[0] = v[0];
        vm[1] = v[1];
        vm[2] = v[2];
        // ---- neighbours at z: row y+1 (z and x components), cell (x0+4, y) (z
        // and y), for the current update of plane z in the next iteration
        if (z < zlast) {
            const unsigned long long pu = p + du;
            const float4 ixu = *reinterpret_cast<const float4*>(I0 + pu);
            const float4 iyu = *reinterpret_cast<const float4*>(I0 + cs + pu);
            const float4 izu = *reinterpret_cast<const float4*>(I0 + 2 * cs + pu);
            const float4 iyu_m = *reinterpret_cast<const float4*>(I0 + cs + pz + du);
            float4 iyu_xm;
            if (x0) iyu_xm = ld4u(I0 + cs + pu - 1);
            else iyu_xm = make_float4(iyu.x, iyu.x, iyu.y, iyu.z);
            const float4 u0z = *reinterpret_cast<const float4*>(V0 + 2 * cs + pu);
            const float4 u0x = *reinterpret_cast<const float4*>(V0 + pu);
            unsigned uu[4] = {0u, 0u, 0u, 0u};
            if (CC) quad_idx(a.kV.idx, pu, uu);
            float4 nu[3];
            float4 c, w;
            quad_coef_n<CC>(a.kV, cs, pu, uu, 2, c, w);
            nu[2] = quad_math(u0z, c, w, quad_curl(iyu, iyu_xm, ixu, ix));
            quad_coef_n<CC>(a.kV, cs, pu, uu, 0, c, w);
            nu[0] = quad_math(u0x, c, w, quad_curl(izu, iz, iyu, iyu_m));
            nu[1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (eub != eue) quad_sources(a.eV, eub, eue, x0, z, 5u, ts, nu);
            vu2m = nu[2];
            vu0m = nu[0];
            const unsigned long long pr = p + dr;
            const float ixr = I0[pr], iyr = I0[cs + pr], izr = I0[2 * cs + pr], ixr_ym = I0[pr - ym];
            const float ixr_m = I0[pz + dr];
            const float r0z = V0[2 * cs + pr], r0y = V0[cs + pr];
            const unsigned ur = CC ? a.kV.idx[pr] : 0u;
            const float2 c2 = coef_n<CC>(a.kV, cs, pr, ur, 2), c1 = coef_n<CC>(a.kV, cs, pr, ur, 1);
            const float c2r = iyr - iy.w - ixr + ixr_ym;
            const float c1r = ixr - ixr_m - izr + iz.w;
            float nrz = r0z * c2.x;
            nrz = nrz + c2.y * c2r;
            float nry = r0y * c1.x;
            nry = nry + c1.y * c1r;
            if (erb != ere) {
                nrz = cell_sources(a.eV, erb, ere, x0 + 4, z, 2, ts, nrz);
                nry = cell_sources(a.eV, erb, ere, x0 + 4, z, 1, ts, nry);
            }
            vr2m = nrz;
            vr1m = nry;
        }
    }
}

// ---------------------------------------------------------------------------
// Tiled quad column sweep (form 3 on meshes of at least 64 quads per row).
// A workgroup is a tile of 64 quads x 4 rows, one wave per row, sweeping a
// z chunk in lock step (one barrier per plane).  The V^{n+1} values the
// current update needs from its neighbours come from the cells' owners: the
// z and x components of row y+1 through LDS (three plane buffers, so one
// barrier per plane separates every write from the reads of the same
// buffer), element 0 of quad x0+4 from the next lane of the wave.  Only the
// tile's top row (wave 3) recomputes row y+1 as k_step4 does, and only lane
// 63 recomputes cell (x0+4, y); the x-1 neighbours of the voltage update
// come from the previous lane and I^n of plane z-1 is carried.  Sources are
// per-quad lists ordered by plane, consumed through cursors.  Arithmetic
// is k_step4's; the Mur faces on x = 0 and x = Nx-1 run their pre and post
// hooks here (below), the other faces' hooks around the launch.  Lanes past
// the mesh run the loop on clamped positions and store nothing.
// ---------------------------------------------------------------------------
constexpr unsigned kQTileRows = kBlock / 64;

// Mur pre and post hooks of point k (coefficients cp, cpp) for face element
// F and neighbour element S of a quad (the MurPre / MurPost hooks' arithmetic):
// y and z from V^n (v0) and V^{n+1} (v); stored when `keep`
template <int F, int S>
__device__ __forceinline__ void mur_fold_quad(const MurFold& M, unsigned k, float cp, float cpp, const float4 v0[3],
                                              const float4 v[3], bool keep, float& fy, float& fz)
{
    float my = f4g(v0[1], S) - cp * f4g(v0[1], F);
    my = my + cp * f4g(v[1], S);
    float mz = f4g(v0[2], S) - cpp * f4g(v0[2], F);
    mz = mz + cpp * f4g(v[2], S);
    if (keep) {
        M.mP[k] = my;
        M.mPP[k] = mz;
    }
    fy = my;
    fz = mz;
}

template <bool CC, bool NT, bool LT>
__global__ __launch_bounds__(kBlock, 3) void k_step4t(const Step4Args ag, const float* __restrict__ V0,
                                                   const float* __restrict__ I0, float* __restrict__ V1,
                                                   float* __restrict__ I1)
{
    extern __shared__ float4 s_tab[];
    __shared__ float4 s_vz[3][kBlock], s_vx[3][kBlock];
    Step4Args a = ag;
    if (LT) {
        stage_table(s_tab, ag.kV.tab, ag.kV.ntab);
        stage_table(s_tab + ag.kV.ntab, ag.kI.tab, ag.kI.ntab);
        __syncthreads();
        a.kV.tab = s_tab;
        a.kI.tab = s_tab + ag.kV.ntab;
    }
    const GridDesc& g = a.g;
    const unsigned long long cs = g.cs;
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned tt = t % a.ntiles, zc = t / a.ntiles;
    const unsigned lane = threadIdx.x & 63u, row = threadIdx.x >> 6;
    const unsigned tqx = tt % a.ntq, tqy = tt / a.ntq;
    const unsigned qx = tqx * 64u + lane, yy = tqy * kQTileRows + row;
    const bool active = qx < a.nq && yy < a.ny;
    // lanes past the mesh compute on a clamped quad and store nothing
    const unsigned x0 = 4u * min(qx, a.nq - 1u), y = min(yy, a.ny - 1u);
    const int ts = (int)a.numts[0];
    const unsigned Nx = g.Nx;
    const unsigned long long plane = g.plane;
    const unsigned z0 = a.za + zc * a.zdepth;
    const unsigned z1 = min(z0 + a.zdepth, a.zb);
    const unsigned zlast = z1 < a.zb ? z1 : z1 - 1;
    const unsigned q = x0 + Nx * y;
    const bool yupd = y + 1 < a.yb;
    const bool xr = x0 + 4 < a.xb;
    const unsigned imask = !active || !yupd ? 0u
                           : xr ? 15u : (x0 + 3 < a.xb ? 7u : x0 + 2 < a.xb ? 3u : x0 + 1 < a.xb ? 1u : 0u);
    const unsigned long long ym = y ? (unsigned long long)Nx : 0ull;
    const unsigned long long du = yupd ? (unsigned long long)Nx : 0ull, dr = xr ? 4ull : 0ull;
    // the top row of the tile recomputes row y+1; lane 63 recomputes (x0+4, y)
    const bool top = row == kQTileRows - 1u;
    const bool edge = lane == 63u && xr;
    const unsigned evb = a.eV.beg[q], eve = a.eV.beg[q + 4];
    const unsigned eib = a.eI.beg[q], eie = a.eI.beg[q + 4];
    const unsigned eub = a.eV.beg[q + du], eue = yupd ? a.eV.beg[q + du + 4] : eub;
    // cell x0+4: the next quad's list (ordered by plane), entries of x0+4 only
    const unsigned erb = a.eV.beg[q + dr], ere = xr ? a.eV.beg[q + dr + 4] : erb;
    // Mur faces on x = 0 and x = Nx-1: the quad holding the face runs their
    // pre and post hooks (Engine_Ext_Mur_ABC::DoPreVoltageUpdates /
    // DoPostVoltageUpdates, engine_ext_mur_abc.cpp:68-142) and uses the value
    // the apply hook will set for the face's y and z components in its own
    // current update; it stores that value too, except on the face's rim,
    // where the other faces' hooks still read or write, and which
    // the MurApply hook sets afterwards
    const bool flo = a.mf[0].on && x0 == 0 && (unsigned)ts >= a.mf[0].start_ts;
    const bool fhi = a.mf[1].on && x0 + 4 == Nx && (unsigned)ts >= a.mf[1].start_ts;
    SrcCursor cv = src_cursor(a.eV, evb, eve, z0), ci = src_cursor(a.eI, eib, eie, z0);
    SrcCursor cu = src_cursor(a.eV, eub, eue, z0);
    float4 vm[3] = {}, vu2m = {}, vu0m = {};
    float vr2m = 0.0f, vr1m = 0.0f;
    // I^n of the own quad at plane z-1, carried from the previous plane
    float4 ixp = {}, iyp = {}, izp = {};
    // and its packed table entries (the engine's two half steps share one
    // index array; read again otherwise)
    uint2 wp = make_uint2(0u, 0u);
    const bool same_idx = a.kI.idx == a.kV.idx;
    if (z0) {
        const unsigned long long p0 = (unsigned long long)(z0 - 1) * plane + q;
        ixp = *reinterpret_cast<const float4*>(I0 + p0);
        iyp = *reinterpret_cast<const float4*>(I0 + cs + p0);
        izp = *reinterpret_cast<const float4*>(I0 + 2 * cs + p0);
    }
    for (unsigned z = z0; z <= zlast; ++z) {
        const unsigned long long p = (unsigned long long)z * plane + q;
        const unsigned long long pz = z ? p - plane : p;
        const unsigned b = z % 3u;
        // Mur coefficients of this plane's face points, issued with the field loads
        float mcp = 0.0f, mcpp = 0.0f, mcpp1 = 0.0f;
        if (flo) {
            mcp = a.mf[0].cP[z * a.ny + y];
            mcpp = a.mf[0].cPP[z * a.ny + y];
            if (top && yupd && z < zlast) mcpp1 = a.mf[0].cPP[z * a.ny + y + 1];
        } else if (fhi) {
            mcp = a.mf[1].cP[z * a.ny + y];
            mcpp = a.mf[1].cPP[z * a.ny + y];
        }
        // ---- own V^{n+1}(x0..x0+3, y, z)
        const float4 ix = *reinterpret_cast<const float4*>(I0 + p);
        const float4 iy = *reinterpret_cast<const float4*>(I0 + cs + p);
        const float4 iz = *reinterpret_cast<const float4*>(I0 + 2 * cs + p);
        // x-1 neighbours of element 0: element 3 of the previous lane's quad;
        // lane 0 reads them (or, at x0 = 0, takes the cell itself)
        float iz_l = __shfl_up(iz.w, 1u, 64), iy_l = __shfl_up(iy.w, 1u, 64);
        if (lane == 0u) {
            iz_l = x0 ? I0[2 * cs + p - 1] : iz.x;
            iy_l = x0 ? I0[cs + p - 1] : iy.x;
        }
        float4 v[3];
        unsigned u[4] = {0u, 0u, 0u, 0u};
        uint2 wv = make_uint2(0u, 0u);
        float fy = 0.0f, fz = 0.0f;        // the face element's y and z after the Mur apply
        {
            const float4 iz_ym = *reinterpret_cast<const float4*>(I0 + 2 * cs + p - ym);
            const float4 ix_ym = *reinterpret_cast<const float4*>(I0 + p - ym);
            const float4 ix_m = z ? ixp : ix;
            const float4 iy_m = z ? iyp : iy;
            const float4 iz_xm = make_float4(iz_l, iz.x, iz.y, iz.z);
            const float4 iy_xm = make_float4(iy_l, iy.x, iy.y, iy.z);
            float4 v0[3];
            v0[0] = ld4<NT>(V0 + p);
            v0[1] = ld4<NT>(V0 + cs + p);
            v0[2] = ld4<NT>(V0 + 2 * cs + p);
            if (CC) {
                wv = *reinterpret_cast<const uint2*>(a.kV.idx + p);
                u[0] = wv.x & 0xFFFFu;
                u[1] = wv.x >> 16;
                u[2] = wv.y & 0xFFFFu;
                u[3] = wv.y >> 16;
            }
            float4 c, w;
            quad_coef_n<CC>(a.kV, cs, p, u, 0, c, w);
            v[0] = quad_math(v0[0], c, w, quad_curl(iz, iz_ym, iy, iy_m));
            quad_coef_n<CC>(a.kV, cs, p, u, 1, c, w);
            v[1] = quad_math(v0[1], c, w, quad_curl(ix, ix_m, iz, iz_xm));
            quad_coef_n<CC>(a.kV, cs, p, u, 2, c, w);
            v[2] = quad_math(v0[2], c, w, quad_curl(iy, iy_xm, ix, ix_ym));
            quad_sources_at(a.eV, cv, x0, z, 7u, ts, v);
            // the hook values are kept for the MurApply hook on the face's rim
            const bool keep = active && z < z1 && (y < 2 || y + 2 >= a.ny || z < 2 || z + 2 >= a.zb);
            if (flo) mur_fold_quad<0, 1>(a.mf[0], z * a.ny + y, mcp, mcpp, v0, v, keep, fy, fz);
            else if (fhi) mur_fold_quad<3, 2>(a.mf[1], z * a.ny + y, mcp, mcpp, v0, v, keep, fy, fz);
        }
        // V^{n+1} as the currents read it: the face element after the Mur apply
        float4 vq1 = v[1], vq2 = v[2];
        if (flo) {
            vq1.x = fy;
            vq2.x = fz;
        } else if (fhi) {
            vq1.w = fy;
            vq2.w = fz;
        }
        if (active && z < z1) {
            // face points off the face's rim (no other face's hook reads or
            // writes them) are stored with the apply's value; the MurApply hook
            // sets the rim after the other faces' post hooks
#pragma unroll
            for (int n = 0; n < 3; ++n) st4<NT>(V1 + n * cs + p, v[n]);
            if ((flo || fhi) && y >= 2 && y + 2 < a.ny && z >= 2 && z + 2 < a.zb) {
                const unsigned long long pf = p + (flo ? 0u : 3u);
                V1[cs + pf] = fy;
                V1[2 * cs + pf] = fz;
            }
        }
        s_vz[b][threadIdx.x] = vq2;
        s_vx[b][threadIdx.x] = v[0];
        // element 0 of the next lane's quad at plane z-1 (cell x0+4)
        const float nr2 = __shfl_down(vm[2].x, 1u, 64);
        const float nr1 = __shfl_down(vm[1].x, 1u, 64);
        __syncthreads();
        // ---- I^{n+1}(x0..x0+3, y, z-1) from the carried plane and v
        if (z > z0 && z < a.zb && imask) {
            const unsigned long long pm = pz;
            unsigned um[4] = {0u, 0u, 0u, 0u};
            if (CC) {
                const uint2 wi = same_idx ? wp : *reinterpret_cast<const uint2*>(a.kI.idx + pm);
                um[0] = wi.x & 0xFFFFu;
                um[1] = wi.x >> 16;
                um[2] = wi.y & 0xFFFFu;
                um[3] = wi.y >> 16;
            }
            float4 u2 = vu2m, u0 = vu0m;
            if (!top) {
                const unsigned bm = (z + 2u) % 3u;     // plane z-1
                u2 = s_vz[bm][threadIdx.x + 64u];
                u0 = s_vx[bm][threadIdx.x + 64u];
            }
            const float r2 = lane == 63u ? vr2m : nr2, r1 = lane == 63u ? vr1m : nr1;
            float4 io[3];
            const float4 vzr = make_float4(vm[2].y, vm[2].z, vm[2].w, r2);
            const float4 vyr = make_float4(vm[1].y, vm[1].z, vm[1].w, r1);
            float4 c, w;
            quad_coef_n<CC>(a.kI, cs, pm, um, 0, c, w);
            io[0] = quad_math(ixp, c, w, quad_curl(vm[2], u2, vm[1], vq1));
            quad_coef_n<CC>(a.kI, cs, pm, um, 1, c, w);
            io[1] = quad_math(iyp, c, w, quad_curl(vm[0], v[0], vm[2], vzr));
            quad_coef_n<CC>(a.kI, cs, pm, um, 2, c, w);
            io[2] = quad_math(izp, c, w, quad_curl(vm[1], vyr, vm[0], u0));
            quad_sources_at(a.eI, ci, x0, z - 1, 7u, ts, io);
            if (imask == 15u) {
#pragma unroll
                for (int n = 0; n < 3; ++n) st4<NT>(I1 + n * cs + pm, io[n]);
            } else {
#pragma unroll
                for (int n = 0; n < 3; ++n)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (imask >> j & 1u) I1[n * cs + pm + j] = f4g(io[n], j);
            }
        }
        vm[0] = v[0];
        vm[1] = vq1;
        vm[2] = vq2;
        ixp = ix;
        iyp = iy;
        izp = iz;
        wp = wv;
        if (z < zlast && top && yupd) {
            // row y+1 at plane z (z and x components), outside the tile
            const unsigned long long pu = p + du;
            const float4 ixu = *reinterpret_cast<const float4*>(I0 + pu);
            const float4 iyu = *reinterpret_cast<const float4*>(I0 + cs + pu);
            const float4 izu = *reinterpret_cast<const float4*>(I0 + 2 * cs + pu);
            const float4 iyu_m = *reinterpret_cast<const float4*>(I0 + cs + pz + du);
            float4 iyu_xm;
            if (x0) iyu_xm = ld4u(I0 + cs + pu - 1);
            else iyu_xm = make_float4(iyu.x, iyu.x, iyu.y, iyu.z);
            const float4 u0z = *reinterpret_cast<const float4*>(V0 + 2 * cs + pu);
            const float4 u0x = *reinterpret_cast<const float4*>(V0 + pu);
            unsigned uu[4] = {0u, 0u, 0u, 0u};
            if (CC) quad_idx(a.kV.idx, pu, uu);
            float4 nu[3];
            float4 c, w;
            quad_coef_n<CC>(a.kV, cs, pu, uu, 2, c, w);
            nu[2] = quad_math(u0z, c, w, quad_curl(iyu, iyu_xm, ixu, ix));
            quad_coef_n<CC>(a.kV, cs, pu, uu, 0, c, w);
            nu[0] = quad_math(u0x, c, w, quad_curl(izu, iz, iyu, iyu_m));
            nu[1] = make_float4(0.f, 0.f, 0.f, 0.f);
            quad_sources_at(a.eV, cu, x0, z, 5u, ts, nu);
            if (flo) {
                // the Mur value of row y+1's face cell (z component)
                float mz1 = u0z.y - mcpp1 * u0z.x;
                mz1 = mz1 + mcpp1 * nu[2].y;
                nu[2].x = mz1;
            }
            vu2m = nu[2];
            vu0m = nu[0];
        }
        if (z < zlast && edge) {
            // cell (x0+4, y) at plane z (z and y components), outside the tile
            const unsigned long long pr = p + dr;
            const float ixr = I0[pr], iyr = I0[cs + pr], izr = I0[2 * cs + pr], ixr_ym = I0[pr - ym];
            const float ixr_m = I0[pz + dr];
            const float r0z = V0[2 * cs + pr], r0y = V0[cs + pr];
            const unsigned ur = CC ? a.kV.idx[pr] : 0u;
            const float2 c2 = coef_n<CC>(a.kV, cs, pr, ur, 2), c1 = coef_n<CC>(a.kV, cs, pr, ur, 1);
            const float c2r = iyr - iy.w - ixr + ixr_ym;
            const float c1r = ixr - ixr_m - izr + iz.w;
            float nrz = r0z * c2.x;
            nrz = nrz + c2.y * c2r;
            float nry = r0y * c1.x;
            nry = nry + c1.y * c1r;
            if (erb != ere) {
                nrz = cell_sources(a.eV, erb, ere, x0 + 4, z, 2, ts, nrz);
                nry = cell_sources(a.eV, erb, ere, x0 + 4, z, 1, ts, nry);
            }
            vr2m = nrz;
            vr1m = nry;
        }
    }
}

// ---------------------------------------------------------------------------
// Two timesteps in one z sweep (k_pair).  The half steps move 38 bytes a cell
// each way through HBM and a single sweep 50 a step; here the intermediate
// state never leaves the chip, so two steps read and write the fields once.
//
// A workgroup owns a tile of tx x ty columns, one per thread, and a z chunk.
// In iteration z four updates run, each a plane behind what it needs from the
// neighbouring columns, so that one barrier a plane serves them all:
//   A  V^{n+1}(z)    from V^n(z), I^n(z), I^n(z-1)       (state n, from memory)
//   B  I^{n+1}(z-1)  from I^n(z-1), V^{n+1}(z-1), V^{n+1}(z)
//   C  V^{n+2}(z-2)  from V^{n+1}(z-2), I^{n+1}(z-2), I^{n+1}(z-3)
//   D  I^{n+2}(z-3)  from I^{n+1}(z-3), V^{n+2}(z-3), V^{n+2}(z-2)
// The own column's planes are carried in registers, the x and y neighbours of
// V^{n+1}(z-1), I^{n+1}(z-2) and V^{n+2}(z-3) come from LDS, double-buffered
// by plane (so the loop body is written twice, by parity).  B needs the next
// column and row, C the previous one, D the next: a tile's results are valid
// on its columns 1 .. tx-3 and rows 1 .. ty-3 (all of them at the mesh
// edges), so tiles advance by tx-3 and ty-3 and recompute their rims; a chunk
// starts one plane early and ends three late.  State n is read from one set
// of buffers (fields, fluxes, timestep counter) and state n+2 written to the
// other.  Per element the arithmetic is volt_tile / curr_tile's, sources
// included, so results are bit-identical.
//
// What bounds it is the round trip of a plane, not bytes or issue: waits
// count outstanding loads in order, so one late gather waits for everything
// in flight.  Hence state n is loaded two planes ahead, and coefficients stay
// in registers until a column's table entry changes.  With loads one plane
// ahead 82 us per step at 253 x 209 x 178 and 321 us at 256^3 with UPML; as
// it is 56 and 218 us, against 149 to 174 and 315 us in two half steps (device
// time per step; 168 and 77 G cells/s, 4.2 and 2.3 TB/s of 50 bytes a cell and
// 52 a UPML position per launch).  Plain stores: non-temporal ones leave the cache
// lines shared by neighbouring tiles to be merged in memory (237 us at 256^3).
// ---------------------------------------------------------------------------
constexpr unsigned kPairMax = 1024;      // threads of a workgroup (columns of its tile)
constexpr unsigned kPairMaxPml = 512;    // with UPML: 202 to 237 registers, without 124 to 128
constexpr unsigned kLdsBytes = 160u * 1024u;   // of a CU
constexpr unsigned kPairLds = 18;        // floats of LDS per column: 3 fields x 3 components x 2 planes

// UPML of k_pair: the slab table in device memory, both sides' arrays
struct PairPml {
    const SlabTab* tab;
    unsigned n;
    unsigned long long npos;
    const unsigned* pidx;
    const float *coefV, *coefI;
    const float4 *ptabV, *ptabI;
};

// sources of one field, in lists per column ordered by plane
constexpr unsigned kSingle = 1u << 31;
struct PairSrc {
    unsigned lo, hi;                     // first and last plane that has any
    // column: first entry and number of entries; marked kSingle where they lie on
    // consecutive planes: first entry, first plane (high half) and number
    const uint2* col;
    ExcArgs ex;
};

struct PairArgs {
    unsigned Nx, Ny, Nz, plane;
    unsigned long long cs;
    unsigned tx, ty, ntx, ntiles;        // tile, tiles along x and over the plane
    unsigned zd;                         // planes per chunk
    CoefArgs kV, kI;
    PairPml pml;
    PairSrc sV, sI;
    const unsigned* tmask;               // bit per tile: its columns hold a source (null: none does)
};

// buffers of one launch: state n read, state n+2 written
struct PairBufs {
    const float *V0, *I0, *fV0, *fI0;
    float *V2, *I2, *fV2, *fI2;
    const unsigned* ts_in;
    unsigned* ts_out;
};

// cursor into the column's list at the first entry from plane z on; NOW: for
// use at plane z only, where the entry's own plane tells whether it is due
template <bool NOW>
__device__ __forceinline__ SrcCursor pair_cursor(const PairSrc& S, unsigned col, unsigned z)
{
    const uint2 q = S.col[col];
    SrcCursor c{q.x & ~kSingle, 0u, ~0u};
    if (q.x & kSingle) {
        const unsigned first = q.y >> 16, n = q.y & 0xFFFFu;
        c.e = c.k + n;
        c.k += z > first ? min(z - first, n) : 0u;
        if (c.k < c.e) c.nz = max(z, first);
        if (NOW) c.e = min(c.e, c.k + 1u);
        return c;
    }
    c.e = c.k + q.y;
    for (unsigned n = q.y; n;) {
        const unsigned h = n / 2;
        if (S.ex.ent[c.k + h].z < z) {
            c.k += h + 1;
            n -= h + 1;
        } else n = h;
    }
    if (c.k < c.e) c.nz = NOW ? z : S.ex.ent[c.k].z;
    return c;
}

// The sources of plane z of the column for one of the four updates, whose
// planes come in order.  CUR: each keeps its cursor in registers; a search at
// every plane is a chain of some eight dependent loads, each of which waits for
// all loads in flight.  Sheets along z with UPML, 160 x 150 x 140: normal to x
// 114 -> 66 us per step, to y 128 -> 76 (half steps 108, 93); 33 x 17 lines in
// 128 x 128 x 96: 43.2 -> 33.9 (39.6).  The kernels of 1024 threads that read
// their coefficients from memory have no register left for cursors (every
// workgroup took 5 to 7 % longer): they find the plane anew, at once in columns
// of one entry a plane (sheet normal to x in a box of 250 x 220 x 180 with 60
// bricks: 210 -> 134, half steps 300), by a search in others.
template <bool CUR>
__device__ __forceinline__ void pair_sources(const PairSrc& S, SrcCursor& c, unsigned col, unsigned z, int ts, float f[3])
{
    if (CUR) col_sources_at(S.ex, c, z, ts, f);
    else if (z >= S.lo && z <= S.hi) {
        SrcCursor n = pair_cursor<true>(S, col, z);
        col_sources_at(S.ex, n, z, ts, f);
    }
}

__device__ __forceinline__ float ldb(const float* __restrict__ b, unsigned off)
{
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(b) + off);
}

__device__ __forceinline__ void stb(float* b, unsigned off, float v)
{
    *reinterpret_cast<float*>(reinterpret_cast<char*>(b) + off) = v;
}

// coefficients of the cell at byte offset off (table entry u)
template <bool CC>
__device__ __forceinline__ void pair_coef(const CoefArgs& k, unsigned long long cs, unsigned off, unsigned u, float a[3],
                                          float b[3])
{
    if (CC) {
        const char* t = reinterpret_cast<const char*>(k.tab) + (u << 5);
        const float4 t0 = *reinterpret_cast<const float4*>(t);
        const float2 t1 = *reinterpret_cast<const float2*>(t + 16);
        a[0] = t0.x; b[0] = t0.y;
        a[1] = t0.z; b[1] = t0.w;
        a[2] = t1.x; b[2] = t1.y;
    } else {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            a[n] = ldb(k.cc + n * cs, off);
            b[n] = ldb(k.cv + n * cs, off);
        }
    }
}

// A copy that the compiler keeps as one.  Merged with its source, a register
// about to be loaded again, it would instead copy (and so wait for) the
// load's result at the end of the loop; and values gathered in a branch are
// waited for there and not after it, where the wait would cover every load
// in flight on the path without the gather too.
template <class V>
__device__ __forceinline__ V keep(V v)
{
    V r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// UPML coefficients of one cell and side
struct PairPmlK {
    float k0[3], ko[3], kn[3];
    unsigned at = ~0u;             // table entry (compressed) or position (plain) they belong to
};

template <int PM>
__device__ __forceinline__ void pair_pml_load(unsigned li, unsigned px, unsigned long long npos, const float* coef,
                                              const float4* ptab, float k[9])
{
    if (PM == kPmlPlain) {
#pragma unroll
        for (int n = 0; n < 9; ++n) k[n] = ldb(coef + n * npos, 4u * li);
    } else {
        const char* t = reinterpret_cast<const char*>(ptab) + 48u * px;
        const float4 t0 = *reinterpret_cast<const float4*>(t), t1 = *reinterpret_cast<const float4*>(t + 16);
        k[0] = t0.x; k[1] = t0.y; k[2] = t0.z;
        k[3] = t0.w; k[4] = t1.x; k[5] = t1.y;
        k[6] = t1.z; k[7] = t1.w; k[8] = *reinterpret_cast<const float*>(t + 32);
    }
}

// one cell's update: x0 its old values, fl its UPML flux (updated), pml: it
// has one.  main: the main update covers it.
template <int PM>
__device__ __forceinline__ void pair_cell(const float x0[3], const float a[3], const float b[3], const float curl[3],
                                          bool pml, const PairPmlK& K, float fl[3], bool main, float out[3])
{
    float f[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const float xin = PM != kNoPml && pml ? fl[n] : x0[n];
        f[n] = xin * a[n];
        f[n] = f[n] + b[n] * curl[n];
        if (!main) f[n] = xin;
    }
    if (PM != kNoPml && pml) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const float t = K.k0[n] * x0[n] - K.ko[n] * fl[n];
            fl[n] = f[n];
            f[n] = t + K.kn[n] * f[n];
        }
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) out[n] = f[n];
}

// the workgroup's sweep; SRC: its columns hold sources
template <int PM, bool CC, bool LT, bool SRC>
__device__ __forceinline__ void pair_sweep(const PairArgs& ag, const PairBufs& B, const CoefArgs& kV, const CoefArgs& kI,
                                           float* s, unsigned tile, unsigned zc, int ts)
{
    const unsigned T = blockDim.x, tid = threadIdx.x;
    const unsigned long long cs = ag.cs, npos = ag.pml.npos;
    const unsigned X0 = tile % ag.ntx * (ag.tx - 3u), Y0 = tile / ag.ntx * (ag.ty - 3u);
    const unsigned ly = tid / ag.tx, lx = tid - ly * ag.tx;
    const bool in = ly < ag.ty && X0 + lx < ag.Nx && Y0 + ly < ag.Ny;
    // threads past the tile or the mesh work on a clamped column and store nothing
    const unsigned x = min(X0 + lx, ag.Nx - 1u), y = min(Y0 + ly, ag.Ny - 1u);
    const bool own = in && (lx || !x) && (ly || !y) && (lx + 2u < ag.tx || X0 + ag.tx >= ag.Nx) &&
                     (ly + 2u < ag.ty || Y0 + ag.ty >= ag.Ny);
    const unsigned col = x + ag.Nx * y;
    const bool cmain = x + 1u < ag.Nx && y + 1u < ag.Ny;
    const unsigned z0 = zc * ag.zd, z1 = min(z0 + ag.zd, ag.Nz), zl = ag.Nz - 1u;
    const unsigned zs = z0 ? z0 - 1u : 0u;                       // first plane of A and B
    const unsigned zA = min(z1 + 1u, zl);                        // last plane of A
    // byte offsets: the column, its x-1 and y-1 neighbours (itself at 0)
    const unsigned P4 = 4u * ag.plane, c4 = 4u * col;
    const unsigned xm = x ? 4u : 0u, ym = y ? 4u * ag.Nx : 0u;
    // the neighbours' LDS slots (the own one where there is no valid neighbour)
    const unsigned nxm = lx ? tid - 1u : tid, nxp = tid + 1u < T ? tid + 1u : tid;
    const unsigned nym = ly ? tid - ag.tx : tid, nyp = tid + ag.tx < T ? tid + ag.tx : tid;
    const float *Vx = B.V0, *Vy = B.V0 + cs, *Vz = B.V0 + 2 * cs, *Ix = B.I0, *Iy = B.I0 + cs, *Iz = B.I0 + 2 * cs;
    // the column's UPML positions up to plane pend: pbase + z * pstep, or none
    unsigned pend = 0, pbase = 0, pstep = 0;
    bool pon = false;
    // state n of the next two planes, by iteration parity: loaded two
    // iterations ahead, for the latency of HBM
    float pv[2][3], pi[2][3], pn[2][4], pf[2][3], qf[2][3];
    unsigned pu[2] = {0, 0}, pl[2] = {~0u, ~0u}, px[2] = {0, 0};
    auto fetch = [&](auto par, unsigned z) {
        constexpr int P = decltype(par)::value;
        const unsigned o = c4 + z * P4;
        if (CC) pu[P] = ag.kV.idx[o >> 2];
        pi[P][0] = ldb(Ix, o);
        pi[P][1] = ldb(Iy, o);
        pi[P][2] = ldb(Iz, o);
        pn[P][0] = ldb(Iz, o - ym);
        pn[P][1] = ldb(Ix, o - ym);
        pn[P][2] = ldb(Iz, o - xm);
        pn[P][3] = ldb(Iy, o - xm);
        pv[P][0] = ldb(Vx, o);
        pv[P][1] = ldb(Vy, o);
        pv[P][2] = ldb(Vz, o);
        if (PM != kNoPml) {
            if (z >= pend) {
                // the slab that holds plane z of the column, and the plane where that changes
                pend = ag.Nz;
                pon = false;
                for (unsigned k = 0; k < ag.pml.n; ++k) {
                    const SlabTab S = ag.pml.tab[k];
                    if ((int)x < S.x0 || (int)x > S.x1 || (int)y < S.y0 || (int)y > S.y1) continue;
                    if ((int)z < S.z0) pend = min(pend, (unsigned)S.z0);
                    else if ((int)z <= S.z1) {
                        pend = (unsigned)S.z1 + 1u;
                        pstep = S.nx * S.ny;
                        pbase = (unsigned)S.off + (x - (unsigned)S.xo) + S.nx * (y - (unsigned)S.y0) - pstep * (unsigned)S.z0;
                        pon = true;
                        break;
                    }
                }
            }
            pl[P] = ~0u;
            if (pon) {
                pl[P] = pbase + z * pstep;
                if (PM == kPmlCompressed) px[P] = ag.pml.pidx[pl[P]];
#pragma unroll
                for (int n = 0; n < 3; ++n) pf[P][n] = ldb(B.fV0 + n * npos, 4u * pl[P]);
            }
        }
    };
    // B's flux of the plane whose position is l
    auto fetch_i = [&](auto par, unsigned l) {
        constexpr int P = decltype(par)::value;
        if (PM != kNoPml && l != ~0u) {
#pragma unroll
            for (int n = 0; n < 3; ++n) qf[P][n] = ldb(B.fI0 + n * npos, 4u * l);
        }
    };
    // carried values, by iteration parity: at iteration z slot P holds
    // V^{n+1}(z-2), I^{n+1}(z-3) and the UPML fluxes of those, slot 1-P
    // V^{n+1}(z-1), I^{n+1}(z-2), V^{n+2}(z-3)
    float v1[2][3] = {}, i1[2][3] = {}, v2[2][3] = {}, i0[3] = {}, fv[2][3], fi[2][3];
    unsigned u1 = 0, u2 = 0, u3 = 0, l1 = ~0u, l2 = ~0u, l3 = ~0u, x1 = 0;
    // coefficients: A's and B's, by parity, serve C and D two iterations later.
    // A column's table entries are gathered only where they change (a material
    // boundary, the graded planes): a gather waits for every load in flight.
    // From an LDS table one set serves all four updates.
    constexpr int S = LT ? 1 : 2;
    float aV[S][3], bV[S][3], aI[S][3], bI[S][3];
    unsigned hV[S], hI[S];
#pragma unroll
    for (int k = 0; k < S; ++k) hV[k] = hI[k] = ~0u;
    PairPmlK kpV[2], kpI[2];
    auto lds_coef = [&](const CoefArgs& k, unsigned u, unsigned& h, float a[3], float b[3]) {
        if (u == h) return;
        h = u;
        pair_coef<true>(k, cs, 0u, u, a, b);
    };
    if (zs) {
        i0[0] = ldb(Ix, c4 + (zs - 1u) * P4);
        i0[1] = ldb(Iy, c4 + (zs - 1u) * P4);
    }
    constexpr bool CUR = PM != kNoPml || LT;
    SrcCursor sA{0u, 0u, ~0u}, sB = sA;
    if (SRC && CUR && ag.sV.col) sA = pair_cursor<false>(ag.sV, col, zs);
    if (SRC && CUR && ag.sI.col) sB = pair_cursor<false>(ag.sI, col, zs);
    SrcCursor sC = sA, sD = sB;
    const std::integral_constant<int, 0> even{};
    const std::integral_constant<int, 1> odd{};
    // (in this order, as in the loop: waits count the loads issued since)
    __builtin_amdgcn_sched_barrier(0);
    fetch(even, zs);
    __builtin_amdgcn_sched_barrier(0);
    fetch(odd, min(zs + 1u, zA));
    fetch_i(odd, pl[0]);
    __builtin_amdgcn_sched_barrier(0);
    // Every iteration runs all four updates: before a plane's first and after
    // its last valid one they work on clamped planes, and nothing reads or
    // stores the result.
    auto iter = [&](auto par, const unsigned z) {
        constexpr int P = decltype(par)::value, Q = 1 - P;
        float* w = s + P * 9u * T + tid;                         // written this iteration
        const float* r = s + Q * 9u * T;                         // written in the previous one
        const unsigned zb = z - 1u, zv = z - 2u, zi = z - 3u;
        const unsigned oa = c4 + min(z, zl) * P4, ob = c4 + min(z ? zb : 0u, zl) * P4;
        const unsigned oc = c4 + min(z > 1u ? zv : 0u, zl) * P4, od = c4 + min(z > 2u ? zi : 0u, zl) * P4;
        float curl[3], i2[3];
        // ---- C: V^{n+2}(z-2)
        {
            if (LT) lds_coef(kV, u2, hV[0], aV[0], bV[0]);
            const float iz_ym = r[5 * T + nym], ix_ym = r[3 * T + nym], iz_xm = r[5 * T + nxm], iy_xm = r[4 * T + nxm];
            const float iy_zm = zv ? i1[P][1] : i1[Q][1], ix_zm = zv ? i1[P][0] : i1[Q][0];
            curl[0] = i1[Q][2] - iz_ym - i1[Q][1] + iy_zm;
            curl[1] = i1[Q][0] - ix_zm - i1[Q][2] + iz_xm;
            curl[2] = i1[Q][1] - iy_xm - i1[Q][0] + ix_ym;
            pair_cell<PM>(v1[P], aV[LT ? 0 : P], bV[LT ? 0 : P], curl, l2 != ~0u, kpV[P], fv[P], true, v2[P]);
            if (SRC) pair_sources<CUR>(ag.sV, sC, col, zv, ts + 1, v2[P]);
        }
        // ---- D: I^{n+2}(z-3)
        {
            if (LT) lds_coef(kI, u3, hI[0], aI[0], bI[0]);
            const float vz_yp = r[8 * T + nyp], vx_yp = r[6 * T + nyp], vz_xp = r[8 * T + nxp], vy_xp = r[7 * T + nxp];
            curl[0] = v2[Q][2] - vz_yp - v2[Q][1] + v2[P][1];
            curl[1] = v2[Q][0] - v2[P][0] - v2[Q][2] + vz_xp;
            curl[2] = v2[Q][1] - vy_xp - v2[Q][0] + vx_yp;
            pair_cell<PM>(i1[P], aI[LT ? 0 : P], bI[LT ? 0 : P], curl, l3 != ~0u, kpI[P], fi[P], cmain && zi < zl, i2);
            if (SRC) pair_sources<CUR>(ag.sI, sD, col, zi, ts + 1, i2);
        }
        if (own && zv >= z0 && zv < z1) {
#pragma unroll
            for (int n = 0; n < 3; ++n) stb(B.V2 + n * cs, oc, v2[P][n]);
            if (PM != kNoPml && l2 != ~0u) {
#pragma unroll
                for (int n = 0; n < 3; ++n) stb(B.fV2 + n * npos, 4u * l2, fv[P][n]);
            }
        }
        if (own && z >= z0 + 3u && zi < z1) {
#pragma unroll
            for (int n = 0; n < 3; ++n) stb(B.I2 + n * cs, od, i2[n]);
            if (PM != kNoPml && l3 != ~0u) {
#pragma unroll
                for (int n = 0; n < 3; ++n) stb(B.fI2 + n * npos, 4u * l3, fi[P][n]);
            }
        }
        // coefficients of A and B, in one round trip
        if (!LT || PM != kNoPml) {
            const bool pA = PM != kNoPml && pl[P] != ~0u, pB = PM != kNoPml && l1 != ~0u;
            const unsigned tA = PM == kPmlPlain ? pl[P] : px[P], tB = PM == kPmlPlain ? l1 : x1;
            const bool gm = !LT && (!CC || pu[P] != hV[LT ? 0 : P] || u1 != hI[LT ? 0 : P]);
            const bool gp = PM != kNoPml && ((pA && tA != kpV[P].at) || (pB && tB != kpI[P].at));
            if (gm || gp) {
                float ca[3], cb[3], da[3], db[3], k[9], q[9];
                if (!LT) {
                    pair_coef<CC>(kV, cs, oa, pu[P], ca, cb);
                    pair_coef<CC>(kI, cs, ob, u1, da, db);
                }
                if (pA) pair_pml_load<PM>(pl[P], px[P], npos, ag.pml.coefV, ag.pml.ptabV, k);
                if (pB) pair_pml_load<PM>(l1, x1, npos, ag.pml.coefI, ag.pml.ptabI, q);
                if (!LT) {
                    hV[LT ? 0 : P] = pu[P];
                    hI[LT ? 0 : P] = u1;
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        aV[LT ? 0 : P][n] = keep(ca[n]);
                        bV[LT ? 0 : P][n] = keep(cb[n]);
                        aI[LT ? 0 : P][n] = keep(da[n]);
                        bI[LT ? 0 : P][n] = keep(db[n]);
                    }
                }
                if (pA) {
                    kpV[P].at = tA;
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        kpV[P].k0[n] = keep(k[n]);
                        kpV[P].ko[n] = keep(k[3 + n]);
                        kpV[P].kn[n] = keep(k[6 + n]);
                    }
                }
                if (pB) {
                    kpI[P].at = tB;
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        kpI[P].k0[n] = keep(q[n]);
                        kpI[P].ko[n] = keep(q[3 + n]);
                        kpI[P].kn[n] = keep(q[6 + n]);
                    }
                }
            }
        }
        // ---- A: V^{n+1}(z)
        {
            if (LT) lds_coef(kV, pu[P], hV[0], aV[0], bV[0]);
            const float iy_zm = z ? i0[1] : pi[P][1], ix_zm = z ? i0[0] : pi[P][0];
            curl[0] = pi[P][2] - pn[P][0] - pi[P][1] + iy_zm;
            curl[1] = pi[P][0] - ix_zm - pi[P][2] + pn[P][2];
            curl[2] = pi[P][1] - pn[P][3] - pi[P][0] + pn[P][1];
            pair_cell<PM>(pv[P], aV[LT ? 0 : P], bV[LT ? 0 : P], curl, pl[P] != ~0u, kpV[P], pf[P], true, v1[P]);
            if (SRC) pair_sources<CUR>(ag.sV, sA, col, z, ts, v1[P]);
        }
        // ---- B: I^{n+1}(z-1)
        {
            if (LT) lds_coef(kI, u1, hI[0], aI[0], bI[0]);
            const float vz_yp = r[2 * T + nyp], vx_yp = r[nyp], vz_xp = r[2 * T + nxp], vy_xp = r[T + nxp];
            curl[0] = v1[Q][2] - vz_yp - v1[Q][1] + v1[P][1];
            curl[1] = v1[Q][0] - v1[P][0] - v1[Q][2] + vz_xp;
            curl[2] = v1[Q][1] - vy_xp - v1[Q][0] + vx_yp;
            pair_cell<PM>(i0, aI[LT ? 0 : P], bI[LT ? 0 : P], curl, l1 != ~0u, kpI[P], qf[P], cmain && zb < zl, i1[P]);
            if (SRC) pair_sources<CUR>(ag.sI, sB, col, zb, ts, i1[P]);
        }
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            w[n * T] = v1[P][n];
            w[(3 + n) * T] = i1[P][n];
            w[(6 + n) * T] = v2[P][n];
            i0[n] = keep(pi[P][n]);
            if (PM != kNoPml) {
                fv[P][n] = keep(pf[P][n]);
                fi[P][n] = keep(qf[P][n]);
            }
        }
        if (LT) {
            u3 = u2;
            u2 = u1;
        }
        u1 = keep(pu[P]);
        if (PM != kNoPml) {
            l3 = l2; l2 = l1; l1 = keep(pl[P]);
            x1 = keep(px[P]);
        }
        fetch(par, min(z + 2u, zA));
        fetch_i(par, pl[Q]);
        __syncthreads();
    };
    // planes zs .. z1+2 (and one past where their number is odd: a mid-loop
    // exit made the compiler copy, and so wait for, the loads just issued)
    for (unsigned z = zs; z <= z1 + 2u; z += 2u) {
        iter(even, z);
        iter(odd, z + 1u);
    }
}

template <int PM, bool CC, bool LT>
__global__ __launch_bounds__(PM == kNoPml ? kPairMax : kPairMaxPml) void k_pair(const PairArgs ag, const PairBufs B)
{
    extern __shared__ float4 s_tab[];
    CoefArgs kV = ag.kV, kI = ag.kI;
    float* s = reinterpret_cast<float*>(s_tab);
    if (LT) {
        stage_table(s_tab, ag.kV.tab, ag.kV.ntab);
        stage_table(s_tab + ag.kV.ntab, ag.kI.tab, ag.kI.ntab);
        kV.tab = s_tab;
        kI.tab = s_tab + ag.kV.ntab;
        s = reinterpret_cast<float*>(s_tab + ag.kV.ntab + ag.kI.ntab);
        __syncthreads();
    }
    const int ts = (int)B.ts_in[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) B.ts_out[0] = (unsigned)ts + 2u;
    const unsigned bid = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned tile = bid % ag.ntiles, zc = bid / ag.ntiles;
    // the leanest sweep for what the workgroup's cells hold
    const bool src = ag.tmask && (ag.tmask[tile >> 5] >> (tile & 31u) & 1u);
    bool pml = false;
    if (PM != kNoPml) {
        const int X0 = (int)(tile % ag.ntx * (ag.tx - 3u)), Y0 = (int)(tile / ag.ntx * (ag.ty - 3u));
        const int za = (int)(zc * ag.zd) - 1, zb = (int)((zc + 1u) * ag.zd) + 1;
        for (unsigned k = 0; k < ag.pml.n; ++k) {
            const SlabTab& S = ag.pml.tab[k];
            pml = pml || (X0 <= S.x1 && X0 + (int)ag.tx > S.x0 && Y0 <= S.y1 && Y0 + (int)ag.ty > S.y0 && za <= S.z1 &&
                          zb >= S.z0);
        }
    }
    if (src) pair_sweep<PM, CC, LT, true>(ag, B, kV, kI, s, tile, zc, ts);
    else if (PM != kNoPml && pml) pair_sweep<PM, CC, LT, false>(ag, B, kV, kI, s, tile, zc, ts);
    else pair_sweep<kNoPml, CC, LT, false>(ag, B, kV, kI, s, tile, zc, ts);
}

// ---------------------------------------------------------------------------
// ++numTS after a single-sweep step (Engine::IterateTS, FDTD/engine.cpp:283).
// Every workgroup of the step reads the counter, so the step itself cannot
// advance it; a one-thread launch after it does, with no fence or atomic
// ordering inside the step.
// ---------------------------------------------------------------------------
__global__ void k_tick(unsigned* __restrict__ numts)
{
    if (threadIdx.x == 0) numts[0] = numts[0] + 1u;
}

// ---------------------------------------------------------------------------
// Mur ABC (Engine_Ext_Mur_ABC, engine_ext_mur_abc.cpp:68-178)
// ---------------------------------------------------------------------------
struct MurDev {
    unsigned na, nb;                      // points along nyP, nyPP
    unsigned long long offP, offPP;       // component offsets nyP*cs, nyPP*cs
    const unsigned* face;                 // [na*nb] linear index of the face point
    const unsigned* shift;                // [na*nb] linear index of the neighbour point
    const float* cP;
    const float* cPP;
    float* mP;
    float* mPP;
    unsigned start_ts;
};

// The current update (curr_tile's arithmetic, FDTD/engine.cpp:170-222) redone
// from the final voltages V1 and the currents of state n, into I1, for the
// quad sweep's currents that read voltages set after the sweep: the planes
// lo..hi along `axis` next to a Mur face, and the cells next to
// a deferred voltage source (k_curr_again).
__device__ __forceinline__ void curr_cell(const GridDesc& g, const float* __restrict__ V1, const float* __restrict__ I0,
                                          float* __restrict__ I1, const CoefArgs& k, unsigned long long p)
{
    const unsigned long long cs = g.cs;
    const unsigned long long dx = 1, dy = g.Nx, dz = g.plane;
    const float* Vx = V1;
    const float* Vy = V1 + cs;
    const float* Vz = V1 + 2 * cs;
    float curl[3];
    curl[0] = Vz[p] - Vz[p + dy] - Vy[p] + Vy[p + dz];
    curl[1] = Vx[p] - Vx[p + dz] - Vz[p] + Vz[p + dx];
    curl[2] = Vy[p] - Vy[p + dx] - Vx[p] + Vx[p + dy];
    float a[3], b[3];
    if (k.idx) {
        const unsigned u = k.idx[p];
        const float4 t0 = k.tab[2 * u], t1 = k.tab[2 * u + 1];
        a[0] = t0.x; b[0] = t0.y;
        a[1] = t0.z; b[1] = t0.w;
        a[2] = t1.x; b[2] = t1.y;
    } else {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            a[m] = k.cc[m * cs + p];
            b[m] = k.cv[m * cs + p];
        }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        float f = I0[m * cs + p] * a[m];
        f = f + b[m] * curl[m];
        I1[m * cs + p] = f;
    }
}

// ---------------------------------------------------------------------------
// lumped RLC (Engine_Ext_LumpedRLC, engine_ext_lumpedRLC.cpp:83-147).  The
// reference rotates its three history buffers once per step (Vd in the pre
// hook, J in the apply hook); after k+1 rotations logical slot i lives in
// buffer (2(k+1) + i) mod 3, so the rotation is derived from numTS.
// ---------------------------------------------------------------------------
struct RlcDev {
    unsigned count;
    const unsigned long long* lin;  // component offset + linear index
    const float* c[9];              // i2v, ilv, vvd, vv2, vj1, vj2, ib0, b1, b2
    float* vd;                      // [3][count]
    float* jn;                      // [3][count]
    float* il;                      // [count]
};

__device__ __forceinline__ unsigned rlc_slot(unsigned ts, unsigned i) { return (2u * ((ts + 1u) % 3u) + i) % 3u; }

// ---------------------------------------------------------------------------
// Lorentz / Drude ADE (engine_ext_lorentzmaterial.cpp:79-173,
// engine_ext_dispersive.cpp:76-132)
// ---------------------------------------------------------------------------
struct LorDev {
    unsigned count;
    const unsigned* lin;   // [count]
    const float* cint;     // [3][count]
    const float* cext;
    const float* clor;     // nullptr: Drude/Debye form
    float* ade;            // [3][count]
    float* lor;            // [3][count]
};

// one term of the ADE current subtracted from a cell's component
struct LorTerm {
    const float* ade;              // the order's [3][count]
    unsigned k, count;
};

// steady-state detection (k_ss_eval)
struct SteadyDev {
    unsigned n, p, cap;
    const unsigned long long* lin;   // [n] component * cs + cell
    float* rec;                      // [n][2p]
    double* state;                   // [0] last max diff, [1] last total energy, [2] evaluations
    unsigned* hist_ts;               // [cap]
    double* hist_diff;               // [cap]
};

// ---------------------------------------------------------------------------
// Extension hooks around the two half steps (FDTD/engine.cpp:224-265).  Each
// hook touches a face or a cell list, microseconds of work, so a step of an
// engine with several extensions is bound by its launches (a small kernel in
// a replayed graph costs 2.5-4.5 us from start to start, whatever it does).
// One launch therefore runs every hook that may run concurrently: the host
// (setup_hooks) keeps the reference's order and opens a new launch only where
// a hook reads or writes a field element that an earlier hook of the launch
// writes.  A workgroup belongs to one job (first[] in the kernel arguments).
// With the hooks before an update beside other work (the currents' after the
// voltage update, the voltages' beside the current update of the step before:
// k_curr_pre), launches and time per step: six Mur faces with steady-state
// detection (96 x 90 x 70) 22 -> 5 and 64.7 -> 26.9 us; Drude, Lorentz and
// Debye boxes with RLC elements (72^3) 17 -> 4 and 38.2 -> 20.3 us; one Mur
// face (27 x 11 x 33) 6 -> 3 and 17.3 -> 11.7 us; 512 x 384 x 320 layers
// around the quad sweep (beside k_curr_again) 0.976 -> 0.934 ms.
//
//   MurPre / MurPost / MurApply  Engine_Ext_Mur_ABC (engine_ext_mur_abc.cpp:68-178);
//                  the faces' applies run in reverse creation order, so where
//                  two faces set one element the face created first wins:
//                  over[] marks, per point and component, the earlier faces
//                  (bit = creation index) that set the element too.
//                  MurPostApply: post and apply of a face in one job, where no
//                  face's apply sets what a post reads
//   RlcPre / RlcApply  Engine_Ext_LumpedRLC (engine_ext_lumpedRLC.cpp:83-147)
//   LorPre / LorApply  Engine_Ext_LorentzMaterial (engine_ext_lorentzmaterial.cpp:79-173,
//                  engine_ext_dispersive.cpp:76-132); the orders' terms of a
//                  cell are subtracted one after another in creation order
//   Excite         Engine_Ext_Excitation (engine_ext_excitation.cpp:33-99): one
//                  thread per (component, cell) group adds its entries in
//                  list order; the current side of the two half steps runs
//                  after the counter advanced (ts_bias -1)
//   SteadyRecord   Engine_Ext_SteadyState's record (engine_ext_steadystate.cpp:50-64)
// ---------------------------------------------------------------------------
enum HookKind { kMurPre, kMurPost, kMurPostApply, kMurApply, kRlcPre, kRlcApply, kLorPre, kLorApply, kExcite, kSteadyRecord };

constexpr unsigned kMaxHookJobs = 12;   // jobs of one launch
constexpr unsigned kMurMaskFaces = 8;   // faces that over[] can name

struct HookJob {
    int kind;
    int curr;                      // the field it works on: 0 voltages, 1 currents
    unsigned n;                    // threads
    MurDev mur;
    const unsigned* list;          // MurApply: the points (null: all)
    const unsigned char* over[2];  // MurApply: earlier faces setting the element (null: none)
    unsigned start[kMurMaskFaces]; // MurApply: first timestep of each face
    RlcDev rlc;
    LorDev lor;
    const unsigned* cell;          // LorApply: cells, their term ranges and terms
    const unsigned* beg;
    const LorTerm* term;
    const unsigned* gbeg;          // Excite
    const unsigned long long* glin;
    const float* amp;
    const unsigned* delay;
    const float* sig;
    unsigned length;
    int period, ts_bias;
    SteadyDev ss;
};

struct HookLaunch {
    const HookJob* jobs;           // device memory
    unsigned n;
    unsigned first[kMaxHookJobs];  // first workgroup of each job
    unsigned nblk;
};

__device__ __forceinline__ bool mur_overset(const HookJob& J, int c, unsigned k, unsigned ts)
{
    if (!J.over[c]) return false;
    const unsigned m = J.over[c][k];
    bool o = false;
#pragma unroll
    for (unsigned j = 0; j < kMurMaskFaces; ++j) o = o || ((m >> j & 1u) && ts >= J.start[j]);
    return o;
}

// the job of the launch's workgroup `bid`, k: the thread within the job
__device__ __forceinline__ const HookJob& hook_job(const HookLaunch& L, unsigned bid, unsigned& k)
{
    unsigned w = 0, f = 0;
#pragma unroll
    for (unsigned i = 1; i < kMaxHookJobs; ++i)
        if (i < L.n && bid >= L.first[i]) {
            w = i;
            f = L.first[i];
        }
    k = (bid - f) * kBlock + threadIdx.x;
    return L.jobs[w];
}

// the hooks before an update: they read F and set the extensions' own values
__device__ __forceinline__ void hook_pre(const HookJob& J, unsigned k, const float* __restrict__ F,
                                         const unsigned long long cs, unsigned ts)
{
    switch (J.kind) {
    case kMurPre: {
        const MurDev& m = J.mur;
        if (ts < m.start_ts) return;
        const unsigned p = m.face[k], s = m.shift[k];
        m.mP[k] = F[m.offP + s] - m.cP[k] * F[m.offP + p];
        m.mPP[k] = F[m.offPP + s] - m.cPP[k] * F[m.offPP + p];
        return;
    }
    case kRlcPre: {
        const RlcDev& r = J.rlc;
        const float* Vd1 = r.vd + rlc_slot(ts, 1) * r.count;
        r.il[k] = r.il[k] + (r.c[0][k] * r.c[1][k]) * Vd1[k];
        return;
    }
    case kLorPre: {                // k = component * count + cell
        const LorDev& d = J.lor;
        const unsigned n = k / d.count;
        const float x = F[n * cs + d.lin[k - n * d.count]];
        const float ade = d.ade[k] * d.cint[k];
        if (d.clor) {
            const float l = d.lor[k] + d.clor[k] * d.ade[k];
            d.lor[k] = l;
            d.ade[k] = ade + d.cext[k] * (x - l);
        } else {
            d.ade[k] = ade + d.cext[k] * x;
        }
        return;
    }
    }
}

// numts: [0] the counter, [1] the timestep of the pre hooks that run beside
// the current update (k_curr_pre): that update advances [0], so the launch
// between the two half steps leaves them the value it will have
__global__ __launch_bounds__(kBlock) void k_hooks(float* __restrict__ V, float* __restrict__ I,
                                                  const unsigned long long cs, const HookLaunch L,
                                                  unsigned* __restrict__ numts)
{
    unsigned k;
    const HookJob& J = hook_job(L, blockIdx.x, k);
    const unsigned ts = numts[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) numts[1] = ts + 1u;
    if (k >= J.n) return;
    float* F = J.curr ? I : V;
    switch (J.kind) {
    case kMurPost:
    case kMurPostApply: {
        const MurDev& m = J.mur;
        if (ts < m.start_ts) return;
        const unsigned s = m.shift[k];
        const float a = m.mP[k] + m.cP[k] * F[m.offP + s];
        const float b = m.mPP[k] + m.cPP[k] * F[m.offPP + s];
        if (J.kind == kMurPost) {
            m.mP[k] = a;
            m.mPP[k] = b;
            return;
        }
        const unsigned p = m.face[k];
        F[m.offP + p] = a;
        F[m.offPP + p] = b;
        return;
    }
    case kMurApply: {
        const MurDev& m = J.mur;
        if (ts < m.start_ts) return;
        if (J.list) k = J.list[k];
        const unsigned p = m.face[k];
        if (!mur_overset(J, 0, k, ts)) F[m.offP + p] = m.mP[k];
        if (!mur_overset(J, 1, k, ts)) F[m.offPP + p] = m.mPP[k];
        return;
    }
    case kRlcApply: {
        const RlcDev& r = J.rlc;
        float* V0 = r.vd + rlc_slot(ts, 0) * r.count;
        const float* V2 = r.vd + rlc_slot(ts, 2) * r.count;
        float* J0 = r.jn + rlc_slot(ts, 0) * r.count;
        const float* J1 = r.jn + rlc_slot(ts, 1) * r.count;
        const float* J2 = r.jn + rlc_slot(ts, 2) * r.count;
        float v = F[r.lin[k]];
        v = r.c[2][k] * (v - r.il[k] + r.c[3][k] * V2[k] + r.c[4][k] * J1[k] + r.c[5][k] * J2[k]);
        V0[k] = v;
        J0[k] = r.c[6][k] * (v - V2[k]) - (r.c[7][k] * r.c[6][k]) * J1[k] - (r.c[8][k] * r.c[6][k]) * J2[k];
        F[r.lin[k]] = v;
        return;
    }
    case kLorApply: {              // k = component * cells + cell
        const unsigned nc = J.n / 3u, n = k / nc, c = k - n * nc;
        const unsigned long long i = n * cs + J.cell[c];
        float x = F[i];
        for (unsigned e = J.beg[c]; e < J.beg[c + 1]; ++e) {
            const LorTerm T = J.term[e];
            x = x - T.ade[n * T.count + T.k];
        }
        F[i] = x;
        return;
    }
    case kExcite: {
        const unsigned long long i = J.glin[k];
        float v = F[i];
        for (unsigned e = J.gbeg[k]; e < J.gbeg[k + 1]; ++e)
            v = v + J.amp[e] * J.sig[exc_sample((int)ts + J.ts_bias, J.delay[e], J.period, J.length)];
        F[i] = v;
        return;
    }
    case kSteadyRecord: {
        const SteadyDev& s = J.ss;
        s.rec[(size_t)k * 2 * s.p + ts % (2 * s.p)] = F[s.lin[k]];
        return;
    }
    default: hook_pre(J, k, F, cs, ts);
    }
}

// ---------------------------------------------------------------------------
// After the hooks of a single-sweep step: the currents of up to six bands of
// planes next to faces and of listed cells again, each a job of workgroups, in
// one launch with the next step's hooks before its voltage update (whose
// voltages are final) and, where no hook follows, the timestep's advance.  The
// sweep writes out of place, so where bands meet the same value is stored
// twice.  One launch each, on 512 x 384 x 320 layers, took 0.955 ms per step,
// this 0.934, of which the sweep is 0.867 and the hooks 0.020.
// ---------------------------------------------------------------------------
constexpr unsigned kMaxBands = 6;  // of one launch

struct CurrBand {
    int axis;
    unsigned lo, hi;               // first and last plane
    unsigned first;                // first workgroup
};

struct CurrAgain {
    CurrBand band[kMaxBands];
    unsigned nband;
    const unsigned long long* cells;   // each with x, y, z below the last line
    unsigned ncells, first;            // of the listed cells
    unsigned nblk;                     // workgroups before the hooks'
};

__device__ __forceinline__ void curr_hooks(const HookLaunch& L, unsigned bid, const float* __restrict__ V,
                                           const unsigned long long cs, const unsigned* __restrict__ numts)
{
    unsigned k;
    const HookJob& J = hook_job(L, bid, k);
    if (k < J.n) hook_pre(J, k, V, cs, numts[1]);
}

__global__ __launch_bounds__(kBlock) void k_curr_again(const GridDesc g, const float* __restrict__ V1,
                                                       const float* __restrict__ I0, float* __restrict__ I1,
                                                       const CoefArgs k, const CurrAgain A, const HookLaunch L,
                                                       unsigned* __restrict__ numts, int tick)
{
    const unsigned bid = blockIdx.x;
    if (bid >= A.nblk) return curr_hooks(L, bid - A.nblk, V1, g.cs, numts);
    if (tick && bid == 0 && threadIdx.x == 0) numts[0] = numts[0] + 1u;
    if (bid >= A.first) {
        const unsigned t = (bid - A.first) * kBlock + threadIdx.x;
        if (t < A.ncells) curr_cell(g, V1, I0, I1, k, A.cells[t]);
        return;
    }
    CurrBand b = A.band[0];
#pragma unroll
    for (unsigned j = 1; j < kMaxBands; ++j)
        if (j < A.nband && bid >= A.band[j].first) b = A.band[j];
    const unsigned d = b.hi - b.lo + 1;
    const unsigned n0 = b.axis == 0 ? d : g.Nx, n1 = b.axis == 1 ? d : g.Ny, n2 = b.axis == 2 ? d : g.Nz;
    const unsigned t = (bid - b.first) * kBlock + threadIdx.x;
    const unsigned r = t / n0, zr = r / n1;
    if (zr >= n2) return;
    const unsigned x = t - r * n0 + (b.axis == 0 ? b.lo : 0u), y = r - zr * n1 + (b.axis == 1 ? b.lo : 0u);
    const unsigned z = zr + (b.axis == 2 ? b.lo : 0u);
    if (x + 1 >= g.Nx || y + 1 >= g.Ny || z + 1 >= g.Nz) return;
    curr_cell(g, V1, I0, I1, k, x + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z);
}

// ---------------------------------------------------------------------------
// The current half step with, in workgroups of their own, the next step's
// hooks before its voltage update: those read voltages, which the current
// update does not set, and values that only voltage hooks use, so they need no
// launch of their own: with it 13.7 us per step at 27 x 11 x 33, 23.0 at 72^3
// and 29.4 at 96 x 90 x 70, without it 11.7, 20.3 and 26.9.  The field accesses
// are the plain ones.
// ---------------------------------------------------------------------------
template <int PM, bool CC>
__global__ __launch_bounds__(kBlock) void k_curr_pre(const GridDesc g, float* I, const float* __restrict__ V,
                                                     const CoefArgs k, const PmlArgs pml, unsigned* __restrict__ numts,
                                                     const unsigned nblk, const HookLaunch L)
{
    if (blockIdx.x >= nblk) return curr_hooks(L, blockIdx.x - nblk, V, g.cs, numts);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(numts, 1u);
    curr_tile<PM, CC, false>(g, xcd_tile(blockIdx.x, nblk), I, V, k, pml);
}

template <int PM, bool CC, bool LT>
__global__ __launch_bounds__(kBlock) void k_curr4_pre(const GridDesc g, const QBoxes boxes, float* I,
                                                      const float* __restrict__ V, const CoefArgs kg, const PmlArgs pml,
                                                      unsigned* __restrict__ numts, const unsigned nblk,
                                                      const HookLaunch L)
{
    if (blockIdx.x >= nblk) return curr_hooks(L, blockIdx.x - nblk, V, g.cs, numts);
    curr4_tile<PM, CC, false, LT>(g, boxes, blockIdx.x, nblk, I, V, kg, pml, numts);
}

// ---------------------------------------------------------------------------
// probes: one block per probe; the terms are gathered in parallel and summed
// by one lane in the reference's order so the result is bit-identical
// (double sum for voltages, float sum for currents).
// ---------------------------------------------------------------------------
struct ProbeDev {
    int type;
    unsigned nelem;
    unsigned off;          // offset into the element tables
    unsigned interval, fd_interval, start_ts, stop_ts, capacity;
    unsigned* count;       // [1]
    unsigned* ts_out;      // [capacity]
    double* val_out;       // [capacity*3]
};

constexpr unsigned kProbeChunk = 2048;

// one probe sample by one workgroup (values gathered in parallel, summed by
// one lane in the reference's term order)
__device__ void probe_block(const ProbeDev P, const float* __restrict__ V, const float* __restrict__ I,
                            const unsigned long long* __restrict__ elin, const signed char* __restrict__ esign,
                            const double* __restrict__ ediv, unsigned ts)
{
    __shared__ float vals[kProbeChunk];
    if (ts < P.start_ts || ts > P.stop_ts) return;
    const bool due = (P.interval && ts % P.interval == 0) || (P.fd_interval && ts % P.fd_interval == 0);
    if (!due) return;
    const float* F = (P.type == EMS_PROBE_CURRENT || P.type == EMS_PROBE_HFIELD) ? I : V;
    double acc_d = 0.0;
    float acc_f = 0.0f;
    double out[3] = {0.0, 0.0, 0.0};
    const bool integral = P.type == EMS_PROBE_VOLTAGE || P.type == EMS_PROBE_CURRENT;
    for (unsigned base = 0; base < P.nelem; base += kProbeChunk) {
        const unsigned m = min(kProbeChunk, P.nelem - base);
        // gathered with the term's sign (a - b and a + (-b) round alike), so
        // the ordered sum below reads nothing from global memory
        for (unsigned e = threadIdx.x; e < m; e += blockDim.x) {
            const unsigned j = P.off + base + e;
            const float v = F[elin[j]];
            vals[e] = integral && esign[j] <= 0 ? -v : v;
        }
        __syncthreads();
        // The ordered sum is a chain of adds; its LDS reads are issued eight
        // at a time, or every term would wait for its own (64^3 cavity, a
        // line of 63 terms: 5.6 -> 4.5 us per sample)
        if (threadIdx.x == 0) {
            if (P.type == EMS_PROBE_VOLTAGE) {
#pragma unroll 8
                for (unsigned e = 0; e < m; ++e) acc_d = acc_d + (double)vals[e];
            } else if (P.type == EMS_PROBE_CURRENT) {
#pragma unroll 8
                for (unsigned e = 0; e < m; ++e) acc_f = acc_f + vals[e];
            } else if (base == 0) {
#pragma unroll
                for (unsigned e = 0; e < 3; ++e) {
                    if (e >= m) break;
                    const double d = ediv[P.off + e];
                    out[e] = d != 0.0 ? (double)vals[e] / d : 0.0;
                }
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned slot = *P.count;
        if (slot < P.capacity) {
            // the three results as plain selects, stored unconditionally
            const double r0 = P.type == EMS_PROBE_VOLTAGE ? acc_d : P.type == EMS_PROBE_CURRENT ? (double)acc_f : out[0];
            const double r1 = integral ? 0.0 : out[1];
            const double r2 = integral ? 0.0 : out[2];
            P.ts_out[slot] = ts;
            P.val_out[3 * slot] = r0;
            P.val_out[3 * slot + 1] = r1;
            P.val_out[3 * slot + 2] = r2;
            *P.count = slot + 1;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_probe(const float* __restrict__ V, const float* __restrict__ I,
                                                  const ProbeDev* __restrict__ probes,
                                                  const unsigned long long* __restrict__ elin,
                                                  const signed char* __restrict__ esign,
                                                  const double* __restrict__ ediv,
                                                  const unsigned* __restrict__ numts)
{
    probe_block(probes[blockIdx.x], V, I, elin, esign, ediv, *numts);
}

// ---------------------------------------------------------------------------
// Batched engine: many independent instances (own mesh, operator, UPML,
// sources, probes) advance together.  Each half step is one persistent
// launch: a workgroup walks the work table (instance, tile) with a stride of
// the grid size; the per-tile arithmetic is that of k_volt / k_curr, so every
// instance is bit-identical to its own engine.
// ---------------------------------------------------------------------------
struct BatchInst {
    GridDesc g;
    float* V;
    float* I;
    CoefArgs kV, kI;
    PmlArgs pV, pI;
    unsigned* numts;
    const float* sig[2];
    unsigned sigLen;
    int period;
    ExcArgs vsrc;                  // voltage sources added by the voltage half step (beg null: by k_batch_excite)
};

template <int PM, bool CC, bool CURR>
__global__ __launch_bounds__(kBlock) void k_batch_half(const BatchInst* __restrict__ inst,
                                                       const uint2* __restrict__ items, unsigned nitems)
{
    for (unsigned w = xcd_tile(blockIdx.x, gridDim.x); w < nitems; w += gridDim.x) {
        const uint2 it = items[w];   // (instance, tile)
        const BatchInst& B = inst[it.x];
        if (CURR) {
            if (it.y == 0 && threadIdx.x == 0) atomicAdd(B.numts, 1u);
            curr_tile<PM, CC, false>(B.g, it.y, B.I, B.V, B.kI, B.pI);
        } else {
            volt_tile<PM, CC, false>(B.g, it.y, B.V, B.I, B.kV, B.pV, B.vsrc, B.numts);
        }
    }
}

// sources of all instances: one thread per (instance, component, cell) group
struct BatchExcGroup {
    unsigned inst;
    unsigned beg, end;             // entries in amp / delay
    unsigned long long lin;        // component * cs + cell
};

__global__ void k_batch_excite(const BatchInst* __restrict__ inst, const BatchExcGroup* __restrict__ grp, unsigned G,
                               const float* __restrict__ amp, const unsigned* __restrict__ delay, int curr, int ts_bias)
{
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= G) return;
    const BatchExcGroup E = grp[g];
    const BatchInst& B = inst[E.inst];
    float* F = curr ? B.I : B.V;
    const float* sig = B.sig[curr];
    const int ts = (int)*B.numts + ts_bias;
    float v = F[E.lin];
    for (unsigned k = E.beg; k < E.end; ++k) v = v + amp[k] * sig[exc_sample(ts, delay[k], B.period, B.sigLen)];
    F[E.lin] = v;
}

// probes of all instances, one workgroup each; a probe not due returns at once
struct BatchProbe {
    ProbeDev P;
    unsigned inst;
    const unsigned long long* elin;
    const signed char* esign;
    const double* ediv;
};

__global__ __launch_bounds__(kBlock) void k_batch_probe(const BatchInst* __restrict__ inst,
                                                        const BatchProbe* __restrict__ probes)
{
    const BatchProbe& Q = probes[blockIdx.x];
    const BatchInst& B = inst[Q.inst];
    probe_block(Q.P, B.V, B.I, Q.elin, Q.esign, Q.ediv, *B.numts);
}

// ---------------------------------------------------------------------------
// field dumps: ProcessFieldsFD::Process (processfields_fd.cpp:72-107, running
// complex<float> sums) and ProcessFieldsTD::Process (processfields_td.cpp:50-91,
// stored samples) of the interpolated E or H field
// (Engine_Interface_FDTD, engine_interface_fdtd.cpp:63-204)
// ---------------------------------------------------------------------------
// A field dump: frequency domain (td = 0; running DFT of the samples) or
// time domain (td = 1; every sample stored).  Samples are taken after the
// steps ts = first + k * fd_interval, k < nsamples.
struct DumpDev {
    unsigned s[3], n[3];          // box start and extent (mesh indices)
    unsigned N[3];
    unsigned fd_interval, nfreq, nsamples;
    unsigned first;               // step of the first sample (0 for frequency-domain dumps)
    int td;
    int field;                    // 0: E from the voltages, 1: H from the currents
    int interp;                   // 0: none, 1: node, 2: cell interpolation
    const float* factors;         // [nsamples][nfreq][2] (frequency domain)
    const double* el[3];          // edge lengths per axis: primary (E) or dual (H)
    float* acc;                   // FD: [nfreq][3][npts][2]; TD: [nsamples][3][npts]
};

__host__ __device__ inline bool dump_sample(const DumpDev& d, unsigned ts, unsigned* k)
{
    if (ts < d.first || (ts - d.first) % d.fd_interval) return false;
    *k = (ts - d.first) / d.fd_interval;
    return *k < d.nsamples;
}

// Engine_Interface_FDTD::GetRawInterpolatedField (E, engine_interface_fdtd.cpp:63-124)
// and GetRawInterpolatedDualField (H, :148-204), component n at node pos, in
// double; without interpolation GetRawField / GetRawDualField (:263-268,
// :134-146), the stored value over its edge length, zero for a zero length.  raw(dx, dy, dz) is component n's stored value at pos + (dx, dy, dz)
// (offsets -1, 0, +1); el: the component's edge lengths (primary for E, dual
// for H).  Shared by the dump kernel and the host-side point read.
template <class Raw>
__host__ __device__ inline double interp_value(int field, int interp, const unsigned* N, const double* el,
                                               const unsigned* pos, int n, Raw raw)
{
    const int nP = (n + 1) % 3, nPP = (n + 2) % 3;
    // the value at pos + sa*e_a + sb*e_b over delta (zero for a zero length)
    auto rv = [&](int a, int sa, int b, int sb, double delta) -> double {
        int o[3] = {0, 0, 0};
        if (a >= 0) o[a] += sa;
        if (b >= 0) o[b] += sb;
        return delta ? (double)raw(o[0], o[1], o[2]) / delta : 0.0;
    };
    const unsigned pn = pos[n];
    if (interp == 0) return rv(-1, 0, -1, 0, el[pn]);
    if (field == 0) {
        if (interp == 1) {
            if (pn == N[n] - 1) return rv(n, -1, -1, 0, el[pn - 1]);
            const double delta = el[pn];
            double out = rv(-1, 0, -1, 0, delta);
            if (delta == 0.0) return 0.0;
            if (pn == 0) return out;
            const double deltaDown = el[pn - 1];
            const double deltaRel = delta / (delta + deltaDown);
            return out * (1.0 - deltaRel) + rv(n, -1, -1, 0, deltaDown) * deltaRel;
        }
        if (pos[0] == N[0] - 1 || pos[1] == N[1] - 1 || pos[2] == N[2] - 1) return 0.0;
        const double delta = el[pn];
        double out = rv(-1, 0, -1, 0, delta);
        out += rv(nP, 1, -1, 0, delta);
        out += rv(nP, 1, nPP, 1, delta);
        out += rv(nPP, 1, -1, 0, delta);
        return out / 4;
    }
    if (interp == 1) {
        if (pos[0] == N[0] - 1 || pos[1] == N[1] - 1 || pos[2] == N[2] - 1 || pos[nP] == 0 || pos[nPP] == 0)
            return 0.0;
        const double delta = el[pn];
        double out = rv(-1, 0, -1, 0, delta);
        out += rv(nP, -1, -1, 0, delta);
        out += rv(nP, -1, nPP, -1, delta);
        out += rv(nPP, -1, -1, 0, delta);
        return out / 4;
    }
    if (pn >= N[n] - 1) return 0.0;
    const double delta = el[pn];
    const double deltaUp = el[pn + 1];
    const double deltaRel = delta / (delta + deltaUp);
    return rv(-1, 0, -1, 0, delta) * (1.0 - deltaRel) + rv(n, 1, -1, 0, deltaUp) * deltaRel;
}

__device__ inline double dump_value(const DumpDev& d, const float* F, unsigned long long cs, const unsigned* pos,
                                    unsigned long long base, const unsigned long long* stride, int n)
{
    const float* C = F + (unsigned long long)n * cs;
    auto raw = [&](int dx, int dy, int dz) -> float {
        long long off = (long long)base;
        off += (long long)dx * (long long)stride[0];
        off += (long long)dy * (long long)stride[1];
        off += (long long)dz * (long long)stride[2];
        return C[off];
    };
    return interp_value(d.field, d.interp, d.N, d.el[n], pos, n, raw);
}

// ProcessFieldsFD::Process (processfields_fd.cpp:72-107): every fd_interval
// steps, field (float) times exp(-2 pi i f T) * 2 dT fd_interval (complex<float>)
// added to the running sum of each frequency.  One thread per dump point.
__global__ void k_fd_dump(const float* __restrict__ F, unsigned long long cs, unsigned Nx, unsigned plane, const DumpDev d,
                          const unsigned* __restrict__ numts)
{
    const unsigned ts = *numts;
    unsigned ks;
    if (!dump_sample(d, ts, &ks)) return;
    const unsigned npts = d.n[0] * d.n[1] * d.n[2];
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= npts) return;
    // dump-box N-I-J-K order: z fastest
    const unsigned lz = k % d.n[2];
    const unsigned ly = (k / d.n[2]) % d.n[1];
    const unsigned lx = k / (d.n[2] * d.n[1]);
    const unsigned pos[3] = {d.s[0] + lx, d.s[1] + ly, d.s[2] + lz};
    const unsigned long long base = pos[0] + (unsigned long long)Nx * pos[1] + (unsigned long long)plane * pos[2];
    const unsigned long long stride[3] = {1ull, (unsigned long long)Nx, (unsigned long long)plane};
    float E[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) E[n] = (float)dump_value(d, F, cs, pos, base, stride, n);
    if (d.td) {
        // ProcessFieldsTD::Process (processfields_td.cpp:50-91): the sample itself
#pragma unroll
        for (int n = 0; n < 3; ++n) d.acc[((unsigned long long)ks * 3 + n) * npts + k] = E[n];
        return;
    }
    for (unsigned f = 0; f < d.nfreq; ++f) {
        const float er = d.factors[(ks * d.nfreq + f) * 2];
        const float ei = d.factors[(ks * d.nfreq + f) * 2 + 1];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            float* a = d.acc + (((unsigned long long)f * 3 + n) * npts + k) * 2;
            a[0] = a[0] + E[n] * er;
            a[1] = a[1] + E[n] * ei;
        }
    }
}

// ---------------------------------------------------------------------------
// Field read-out: component planes x0 .. x0+nx-1 of one component, [z][y][x]
// on the device, as [x][y][z].  A workgroup turns one 32 x 32 tile of x and z
// at one y through LDS, so that both sides move whole cache lines and the
// copy to the host lands in the caller's array (a staged copy and a threaded
// host loop, writing single floats Ny * Nz apart, before: both fields of
// 64^3 lines 2.9 ms, of 47^3 1.2 ms more).
// ---------------------------------------------------------------------------
constexpr unsigned kTurn = 32;
__global__ __launch_bounds__(kTurn * 8) void k_to_nijk(const float* __restrict__ src, float* __restrict__ dst,
                                                       unsigned Nx, unsigned Ny, unsigned Nz, unsigned x0, unsigned nx)
{
    __shared__ float t[kTurn][kTurn + 1];
    const unsigned lx = threadIdx.x % kTurn, ly = threadIdx.x / kTurn;
    const unsigned bx = blockIdx.x * kTurn, bz = blockIdx.y * kTurn;
    for (unsigned y = blockIdx.z; y < Ny; y += gridDim.z) {
        for (unsigned k = ly; k < kTurn; k += 8) {
            const unsigned x = bx + lx, z = bz + k;
            if (x < nx && z < Nz) t[k][lx] = src[x0 + x + (size_t)Nx * (y + (size_t)Ny * z)];
        }
        __syncthreads();
        for (unsigned k = ly; k < kTurn; k += 8) {
            const unsigned x = bx + k, z = bz + lx;
            if (x < nx && z < Nz) dst[((size_t)x * Ny + y) * Nz + z] = t[lx][k];
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// energy (Engine_Interface_FDTD::CalcFastEnergy): per-block double partials
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_energy(const float* __restrict__ V, const float* __restrict__ I,
                                                   unsigned long long cs, unsigned Nx, unsigned Ny, unsigned Nz,
                                                   double* __restrict__ part)
{
    __shared__ double se[kBlock], sh[kBlock];
    const unsigned long long plane = (unsigned long long)Nx * Ny;
    const unsigned long long tot = plane * Nz;
    double e = 0.0, h = 0.0;
    for (unsigned long long p = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; p < tot;
         p += (unsigned long long)gridDim.x * blockDim.x) {
        const unsigned long long z = p / plane;
        const unsigned long long r = p - z * plane;
        const unsigned long long y = r / Nx, x = r - y * Nx;
        if (x + 1 >= Nx || y + 1 >= Ny || z + 1 >= Nz) continue;
        for (int n = 0; n < 3; ++n) {
            const double v = V[n * cs + p], c = I[n * cs + p];
            e += v * v;
            h += c * c;
        }
    }
    se[threadIdx.x] = e;
    sh[threadIdx.x] = h;
    __syncthreads();
    for (unsigned s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            se[threadIdx.x] += se[threadIdx.x + s];
            sh[threadIdx.x] += sh[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = se[0];
        part[2 * blockIdx.x + 1] = sh[0];
    }
}

// one thread: the energy from k_energy's partial sums, summed in workgroup
// order (as ems_energy sums them on the host)
__global__ void k_energy_total(const double* __restrict__ part, unsigned nb, double* __restrict__ out)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double e = 0.0, m = 0.0;
    for (unsigned b = 0; b < nb; ++b) {
        e += part[2 * b];
        m += part[2 * b + 1];
    }
    *out = 8.85418781762e-12 * e + 1.256637062e-6 * m;
}

}  // namespace

// Workgroups of the energy reduction, and the device scratch of the
// allocation-free energy entry point (ems_energy_noalloc): the partial sums
// of those workgroups, two doubles each (16 KiB; every device the library runs
// on holds one copy until the process ends).  Host code never passes the
// array's name to a kernel or a copy: it uses the per-device address from
// hipGetSymbolAddress (scratch_setup).
constexpr unsigned kEnergyBlocks = 1024;
static __device__ __align__(256) double scratch[2 * kEnergyBlocks];

namespace {

// ---------------------------------------------------------------------------
// Adjoint of the timestep (discrete adjoint of the two half steps with UPML),
// for gradients of a DFT-of-probe objective with respect to the coefficients.
// Forward half step of one cell (n = x, y, z), curl c, UPML flux F:
//   plain: X' = cc*X + cv*c
//   UPML : f = cc*F + cv*c;  X' = c0*X - cfo*F + cfn*f;  F' = f
// The transposed half step maps the adjoint (lX', lF') of the new state to
// the adjoint of the old state and the adjoint of the curl:
//   plain: lX = cc*lX';  lc = cv*lX'
//   UPML : lf = lF' + cfn*lX';  lX = c0*lX';  lF = -cfo*lX' + cc*lf;  lc = cv*lf
// and lc is scattered back through the transposed curl, evaluated here in
// gather form (terms whose forward index clamps to the cell itself vanish,
// as the forward curl cancels there).
// ---------------------------------------------------------------------------
struct AdjBox {
    unsigned x0, y0, z0, nx, ny, nz;   // inclusive-exclusive box of edges
    unsigned long long n;              // nx*ny*nz
};

__device__ __forceinline__ bool in_adj_box(const AdjBox& b, unsigned x, unsigned y, unsigned z, unsigned long long& k)
{
    if (x < b.x0 || y < b.y0 || z < b.z0 || x >= b.x0 + b.nx || y >= b.y0 + b.ny || z >= b.z0 + b.nz) return false;
    k = (x - b.x0) + (unsigned long long)b.nx * ((y - b.y0) + (unsigned long long)b.ny * (z - b.z0));
    return true;
}

// UPML coefficients c0, cfo, cfn of position li
template <int PM>
__device__ __forceinline__ void pml_coefs(const PmlArgs& P, unsigned long long li, float k0[3], float ko[3], float kn[3])
{
    if (PM == kPmlPlain) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            k0[n] = P.coef[n * P.npos + li];
            ko[n] = P.coef[(3 + n) * P.npos + li];
            kn[n] = P.coef[(6 + n) * P.npos + li];
        }
    } else {
        const unsigned u = P.pidx[li];
        const float4 t0 = P.ptab[3 * u], t1 = P.ptab[3 * u + 1], t2 = P.ptab[3 * u + 2];
        k0[0] = t0.x; k0[1] = t0.y; k0[2] = t0.z;
        ko[0] = t0.w; ko[1] = t1.x; ko[2] = t1.y;
        kn[0] = t1.z; kn[1] = t1.w; kn[2] = t2.x;
    }
}

// objective probes: F_p += (V[lin_p] / div_p) * w, w = exp(-2 pi i f t) * dT
// at t = ts*dT (voltages after step ts)
struct AdjProbe {
    unsigned long long lin;
    double div;
};

// adjoint source of J = sum |F_p|^2 at step ts: dJ/dV = 2 Re(conj(F) w) / div
struct AdjSrc {
    float* lV;
    const AdjProbe* pr;
    unsigned np;
    double f, dT;
    unsigned ts;
    const double* F;
};

__device__ __forceinline__ void adj_source(const AdjSrc& s, unsigned p)
{
    if (p >= s.np) return;
    const double t = (double)s.ts * s.dT;
    const double ph = -2.0 * 3.141592653589793238462643383279 * s.f * t;
    const double g = 2.0 * (s.F[2 * p] * cos(ph) * s.dT + s.F[2 * p + 1] * sin(ph) * s.dT) / s.pr[p].div;
    s.lV[s.pr[p].lin] = (float)((double)s.lV[s.pr[p].lin] + g);
}

// transposed current half step, one thread per (x, y) column sweeping z.
// lI' = lI + curl_I^T(B) (B: curl adjoint left by the transposed voltage
// half step of the later timestep); writes lI, lFI and A = curl_V adjoint.
// The workgroups past the mesh's add the adjoint source of this step's
// objective to the voltages' adjoint, which this half step does not touch (a
// launch of its own took 3.2 us of 31).
template <int PM, bool CC>
__global__ __launch_bounds__(kBlock) void k_adj_curr(const GridDesc g, float* __restrict__ lI,
                                                     const float* __restrict__ B, float* __restrict__ A,
                                                     const CoefArgs k, const PmlArgs pml, float* __restrict__ lFI,
                                                     unsigned nblk, const AdjSrc src)
{
    if (blockIdx.x >= nblk) {
        adj_source(src, (blockIdx.x - nblk) * kBlock + threadIdx.x);
        return;
    }
    const unsigned t = xcd_tile(blockIdx.x, nblk);
    const unsigned qt = t % g.qtiles, zc = t / g.qtiles;
    unsigned x, y;
    if (!tile_column(g, qt, x, y)) return;
    const unsigned z0 = zc * g.zdepth, z1 = min(z0 + g.zdepth, g.Nz);
    const unsigned long long cs = g.cs;
    const unsigned Nx = g.Nx;
    const bool col_upd = x + 1 < g.Nx && y + 1 < g.Ny;
    const unsigned pcm = PM != kNoPml ? pml_colmask(pml, (int)x, (int)y) : 0u;
    for (unsigned z = z0; z < z1; ++z) {
        const unsigned long long p = x + (unsigned long long)Nx * y + (unsigned long long)g.plane * z;
        // lI' = lI + curl_I^T(B); curl_I of the voltage update uses lower
        // neighbours, clamped to the cell itself at index 0
        float l[3];
        {
            const float* B0 = B;
            const float* B1 = B + cs;
            const float* B2 = B + 2 * cs;
            float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
            if (z > 0) { s0 += B1[p]; s1 -= B0[p]; }
            if (z + 1 < g.Nz) { s0 -= B1[p + g.plane]; s1 += B0[p + g.plane]; }
            if (y > 0) { s0 -= B2[p]; s2 += B0[p]; }
            if (y + 1 < g.Ny) { s0 += B2[p + Nx]; s2 -= B0[p + Nx]; }
            if (x > 0) { s1 += B2[p]; s2 -= B1[p]; }
            if (x + 1 < g.Nx) { s1 -= B2[p + 1]; s2 += B1[p + 1]; }
            l[0] = lI[p] + s0;
            l[1] = lI[cs + p] + s1;
            l[2] = lI[2 * cs + p] + s2;
        }
        const bool upd = col_upd && z + 1 < g.Nz;
        float lo[3], a[3] = {0.0f, 0.0f, 0.0f};
        unsigned li = 0;
        const bool in_pml = PM != kNoPml && pcm && pml_at_col(pml, pcm, (int)x, (int)y, (int)z, li);
        if (upd) {
            float ca[3], cb[3];
            load_coef<CC>(k, cs, p, CC ? k.idx[p] : 0u, ca, cb);
            if (in_pml) {
                float k0[3], ko[3], kn[3];
                pml_coefs<PM>(pml, li, k0, ko, kn);
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    const float lf = lFI[n * pml.npos + li] + kn[n] * l[n];
                    lo[n] = k0[n] * l[n];
                    lFI[n * pml.npos + li] = ca[n] * lf - ko[n] * l[n];
                    a[n] = cb[n] * lf;
                }
            } else {
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    lo[n] = ca[n] * l[n];
                    a[n] = cb[n] * l[n];
                }
            }
        } else if (in_pml) {
            // UPML hooks alone: X' = c0*X + (cfn - cfo)*F, F' = F
            float k0[3], ko[3], kn[3];
            pml_coefs<PM>(pml, li, k0, ko, kn);
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                lo[n] = k0[n] * l[n];
                lFI[n * pml.npos + li] = lFI[n * pml.npos + li] + (kn[n] - ko[n]) * l[n];
            }
        } else {
#pragma unroll
            for (int n = 0; n < 3; ++n) lo[n] = l[n];
        }
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            lI[n * cs + p] = lo[n];
            A[n * cs + p] = a[n];
        }
    }
}

// transposed voltage half step: lV' = lV + curl_V^T(A); writes lV, lFV,
// B = curl_I adjoint, and accumulates dJ/dvi, dJ/dvv on the box edges from
// the recorded forward curl and voltage of the step.
template <int PM, bool CC>
__global__ __launch_bounds__(kBlock) void k_adj_volt(const GridDesc g, float* __restrict__ lV,
                                                     const float* __restrict__ A, float* __restrict__ B,
                                                     const CoefArgs k, const PmlArgs pml, float* __restrict__ lFV,
                                                     const AdjBox box, const float* __restrict__ hc,
                                                     const float* __restrict__ hv, double* __restrict__ gvi,
                                                     double* __restrict__ gvv)
{
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned qt = t % g.qtiles, zc = t / g.qtiles;
    unsigned x, y;
    if (!tile_column(g, qt, x, y)) return;
    const unsigned z0 = zc * g.zdepth, z1 = min(z0 + g.zdepth, g.Nz);
    const unsigned long long cs = g.cs;
    const unsigned Nx = g.Nx;
    const unsigned pcm = PM != kNoPml ? pml_colmask(pml, (int)x, (int)y) : 0u;
    for (unsigned z = z0; z < z1; ++z) {
        const unsigned long long p = x + (unsigned long long)Nx * y + (unsigned long long)g.plane * z;
        // lV' = lV + curl_V^T(A); curl_V of the current update uses upper
        // neighbours, A is zero where the current update does not run
        float l[3];
        {
            const float* A0 = A;
            const float* A1 = A + cs;
            const float* A2 = A + 2 * cs;
            float s0 = A1[p] - A2[p];
            float s1 = A2[p] - A0[p];
            float s2 = A0[p] - A1[p];
            if (z > 0) { s0 -= A1[p - g.plane]; s1 += A0[p - g.plane]; }
            if (y > 0) { s0 += A2[p - Nx]; s2 -= A0[p - Nx]; }
            if (x > 0) { s1 -= A2[p - 1]; s2 += A1[p - 1]; }
            l[0] = lV[p] + s0;
            l[1] = lV[cs + p] + s1;
            l[2] = lV[2 * cs + p] + s2;
        }
        float ca[3], cb[3], lo[3], b[3];
        load_coef<CC>(k, cs, p, CC ? k.idx[p] : 0u, ca, cb);
        unsigned li = 0;
        const bool in_pml = PM != kNoPml && pcm && pml_at_col(pml, pcm, (int)x, (int)y, (int)z, li);
        if (in_pml) {
            float k0[3], ko[3], kn[3];
            pml_coefs<PM>(pml, li, k0, ko, kn);
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                const float lf = lFV[n * pml.npos + li] + kn[n] * l[n];
                lo[n] = k0[n] * l[n];
                lFV[n * pml.npos + li] = ca[n] * lf - ko[n] * l[n];
                b[n] = cb[n] * lf;
            }
        } else {
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                lo[n] = ca[n] * l[n];
                b[n] = cb[n] * l[n];
            }
            unsigned long long kb;
            if (in_adj_box(box, x, y, z, kb)) {
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    gvi[n * box.n + kb] += (double)l[n] * (double)hc[n * box.n + kb];
                    gvv[n * box.n + kb] += (double)l[n] * (double)hv[n * box.n + kb];
                }
            }
        }
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            lV[n * cs + p] = lo[n];
            B[n * cs + p] = b[n];
        }
    }
}

// After a forward step (and before the first): the running DFT of the
// objective probes (last workgroups, np = 0 before the first step) and, where
// hc is given, the forward curl of the currents and the voltages on the box
// edges, the inputs of the coming voltage update.
__global__ __launch_bounds__(kBlock) void k_adj_sample(const GridDesc g, const float* __restrict__ V,
                                                       const float* __restrict__ I, const AdjBox box,
                                                       float* __restrict__ hc, float* __restrict__ hv, unsigned rblk,
                                                       const AdjProbe* __restrict__ pr, unsigned np, double f, double dT,
                                                       const unsigned* __restrict__ numts, double* __restrict__ F)
{
    if (blockIdx.x >= rblk) {
        const unsigned q = (blockIdx.x - rblk) * kBlock + threadIdx.x;
        if (q >= np) return;
        const double t = (double)*numts * dT;
        const double ph = -2.0 * 3.141592653589793238462643383279 * f * t;
        const double v = (double)V[pr[q].lin] / pr[q].div;
        F[2 * q] += v * cos(ph) * dT;
        F[2 * q + 1] += v * sin(ph) * dT;
        return;
    }
    const unsigned long long kk = blockIdx.x * (unsigned long long)kBlock + threadIdx.x;
    if (kk >= box.n) return;
    const unsigned x = box.x0 + (unsigned)(kk % box.nx);
    const unsigned y = box.y0 + (unsigned)((kk / box.nx) % box.ny);
    const unsigned z = box.z0 + (unsigned)(kk / ((unsigned long long)box.nx * box.ny));
    const unsigned long long cs = g.cs;
    const unsigned long long p = x + (unsigned long long)g.Nx * y + (unsigned long long)g.plane * z;
    const unsigned long long xm = x ? 1 : 0, ym = y ? g.Nx : 0, zm = z ? g.plane : 0;
    const float* Ix = I;
    const float* Iy = I + cs;
    const float* Iz = I + 2 * cs;
    hc[kk] = Iz[p] - Iz[p - ym] - Iy[p] + Iy[p - zm];
    hc[box.n + kk] = Ix[p] - Ix[p - zm] - Iz[p] + Iz[p - xm];
    hc[2 * box.n + kk] = Iy[p] - Iy[p - xm] - Ix[p] + Ix[p - ym];
#pragma unroll
    for (int n = 0; n < 3; ++n) hv[n * box.n + kk] = V[n * cs + p];
}

// ---------------------------------------------------------------------------
// steady-state detection (Engine_Ext_SteadyState::Apply2Voltages,
// FDTD/extensions/engine_ext_steadystate.cpp:50-107).  Priority +2e6: it runs
// before every other apply hook, on the voltages of the completed voltage
// update.  Every step records the probe voltages at TS % 2p; at TS % p == 0,
// TS >= 2p it compares the last two periods and the energy change.
// ---------------------------------------------------------------------------
// The reference's evaluation, one workgroup of kSsThreads.  The last wave's
// first two lanes sum k_energy's partials, the other lanes a probe's power
// and change each, every sum in the reference's order; the maxima do not
// depend on theirs.  (One thread for all of it: 445 us, a serial chain of
// some 4000 dependent loads, against 46 us; 96 x 90 x 70 box, 21 probes.)
constexpr unsigned kSsThreads = 256;
__global__ __launch_bounds__(kSsThreads) void k_ss_eval(const SteadyDev s, const double* __restrict__ part, unsigned nb,
                                                        const unsigned* __restrict__ numts)
{
    constexpr unsigned kProbeThreads = kSsThreads - 64;
    __shared__ double s_sum[2], s_max[kProbeThreads];
    __shared__ int s_any[kProbeThreads];
    const unsigned t = threadIdx.x;
    const unsigned TS = *numts, p = s.p;
    const unsigned rel_pos = TS % (2 * p);
    unsigned old_pos = 0, new_pos = p;
    if (rel_pos <= p) {
        new_pos = 0;
        old_pos = p;
    }
    if (t < kProbeThreads) {
        double most = 0;
        for (unsigned n = t; n < s.n; n += kProbeThreads) {
            const float* buf = s.rec + (size_t)n * 2 * p + new_pos;
            double cp = 0;
#pragma unroll 8
            for (unsigned nt = 0; nt < p; ++nt) cp += (double)buf[nt] * (double)buf[nt];
            most = fmax(most, cp);
        }
        s_max[t] = most;
    } else if (t < kProbeThreads + 2) {
        const double* q = part + (t - kProbeThreads);
        double e = 0;
#pragma unroll 8
        for (unsigned b = 0; b < nb; ++b) e += q[2 * b];
        s_sum[t - kProbeThreads] = e;
    }
    __syncthreads();
    double max_pow = 0;
    for (unsigned n = 0; n < min(s.n, kProbeThreads); ++n) max_pow = fmax(max_pow, s_max[n]);
    __syncthreads();
    if (t < kProbeThreads) {
        double diff = 0;
        int any = 0;
        for (unsigned n = t; n < s.n; n += kProbeThreads) {
            const float* bn = s.rec + (size_t)n * 2 * p + new_pos;
            const float* bo = s.rec + (size_t)n * 2 * p + old_pos;
            double cp = 0, dp = 0;
#pragma unroll 8
            for (unsigned nt = 0; nt < p; ++nt) {
                const double a = bn[nt], b = bo[nt];
                cp += a * a;
                dp += (b - a) * (b - a);
            }
            if (cp > max_pow * 1e-2) {
                diff = fmax(diff, dp / cp);
                any = 1;
            }
        }
        s_max[t] = diff;
        s_any[t] = any;
    }
    __syncthreads();
    if (t != 0) return;
    const double curr_total_energy = 8.85418781762e-12 * s_sum[0] + 1.256637062e-6 * s_sum[1];
    bool no_valid = true;
    double last_max_diff = 0;
    const double last_total_energy = s.state[1];
    if (last_total_energy > 0) {
        last_max_diff = fabs(curr_total_energy - last_total_energy) / last_total_energy;
        no_valid = false;
    }
    for (unsigned n = 0; n < min(s.n, kProbeThreads); ++n)
        if (s_any[n]) {
            last_max_diff = fmax(last_max_diff, s_max[n]);
            no_valid = false;
        }
    if (no_valid || last_max_diff > 1) last_max_diff = 1;
    s.state[0] = last_max_diff;
    s.state[1] = curr_total_energy;
    const unsigned k = (unsigned)s.state[2];
    if (k < s.cap) {
        s.hist_ts[k] = TS;
        s.hist_diff[k] = last_max_diff;
    }
    s.state[2] = (double)(k + 1);
}

template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
};

void parallel_rows(size_t n, const std::function<void(size_t, size_t)>& fn);

}  // namespace

// ---------------------------------------------------------------------------
// engine state
// ---------------------------------------------------------------------------
struct ems_engine;

// Device memory for engine h or what works on it.  Where there is none left,
// the read-out's buffer and the ones that only pairs of timesteps need make room.
static hipError_t device_malloc(ems_engine* h, void** q, size_t bytes);

struct ems_engine {
    int device = 0;
    hipStream_t stream = nullptr;
    GridDesc g{};
    unsigned N[3] = {0, 0, 0};
    unsigned long long cs = 0;
    float *V = nullptr, *I = nullptr;          // current state
    float *V_alt = nullptr, *I_alt = nullptr;  // second buffers of the fused step (state n+1)
    float* V_base = nullptr;                   // V at set-up (buffer parity of the fused step)
    // coefficient layout: plain arrays or per-cell index + tables
    int layout_req = EMS_LAYOUT_AUTO;
    bool cmp = false;
    float *vv = nullptr, *vi = nullptr, *ii = nullptr, *iv = nullptr;
    unsigned short* cidx = nullptr;
    float* ctab[2] = {nullptr, nullptr};
    unsigned n_unique = 0;
    CoefArgs kV{}, kI{};
    unsigned* numts_dev = nullptr;        // [0] the counter, [1] see k_hooks
    unsigned numTS = 0;
    bool inited = false;
    bool async = false;
    struct Alloc {
        void* p;
        size_t bytes;
    };
    std::vector<Alloc> allocs;
    size_t alloc_bytes = 0, alloc_most = ~(size_t)0;      // device memory in use, its limit (EMS_DEVICE_BYTES)
    bool room(size_t bytes) const { return alloc_bytes <= alloc_most && bytes <= alloc_most - alloc_bytes; }

    // excitation: entries grouped per (component, cell), each group in list order
    struct Exc {
        unsigned K = 0, G = 0;
        unsigned* gbeg = nullptr;         // [G + 1]
        unsigned long long* glin = nullptr;   // [G] component * cs + cell
        float* amp = nullptr;             // [K] in group order
        unsigned* delay = nullptr;        // [K]
        std::vector<ExcEnt> host;         // list order, for the fused step's tile lists
        std::vector<unsigned> h_gbeg;      // host copies of the groups (batched engine)
        std::vector<unsigned long long> h_glin;
        std::vector<float> h_amp;
        std::vector<unsigned> h_delay;
    } exc[2];
    float* sig[2] = {nullptr, nullptr};
    unsigned sigLen = 0;
    int period = 0;
    bool has_exc = false;

    // UPML: host staging per slab until init
    struct SlabHost {
        SlabTab tab;
        unsigned num[3] = {0, 0, 0};      // slab extent (mesh lines)
        unsigned long long cnt = 0;       // cells of the slab
        std::vector<float> v[3], i[3];   // vv, vvfo, vvfn / ii, iifo, iifn, [3][cnt] x-fastest
    };
    std::vector<SlabHost> slabs;
    PmlArgs pmlV{}, pmlI{};
    float* flux_alt[2] = {nullptr, nullptr};   // second flux buffers of the fused step (V, I)
    // fused single-sweep step
    int fused_req = -1;                   // -1 auto, 0 two half steps, 1 LDS sweep, 2 column sweep, 3 quad sweep
    int fused = 0;                        // active form: 0 two half steps, 1 k_step, 2 k_step2
    bool nt_fields = false;               // non-temporal own-field accesses in the half steps
    int quad_req = -1;                    // -1 auto, 0 one cell per lane, 1 quads (four x cells per lane)
    bool lds_tab = false;                 // quad kernels read the compressed tables from LDS
    bool quad = false;                    // the half steps run k_volt4 / k_curr4
    GridDesc gq{};                        // z depth of the quad half steps
    // quad boxes: the whole mesh, or on a UPML mesh the box without UPML
    // cells (qbox_in, launched without UPML code) and the boxes around it
    QBoxes qbox_all{}, qbox_in{}, qbox_out{};
    unsigned qblk_all = 0, qblk_in = 0, qblk_out = 0;
    QBox* qbox_dev = nullptr;             // the three box lists, kMaxQBoxes each
    // voltage sources added by k_volt4 / k_volt (per-quad or per-column lists;
    // beg null: the Excite hook adds them)
    ExcArgs qsrc{};
    bool qsplit = false;
    unsigned ntx = 0, nty = 0, fzdepth = 0, fnzc = 0;
    bool q4tile = false;                  // form 3 runs k_step4t (64 x 4 quad tiles)
    unsigned q4ntq = 0;                   // its tiles along x
    int mur_fold[2] = {-1, -1};           // Mur faces (index) on x = 0 / x = Nx-1 whose pre and post hooks k_step4t runs
    unsigned* mur_rim[2] = {nullptr, nullptr};    // their rim points (y or z within 2 lines of the mesh edge)
    unsigned nrim[2] = {0, 0};
    ExcArgs eV{}, eI{};
    // two timesteps per launch (k_pair) where no sample falls between them;
    // the arguments that stay the same, the second timestep counter
    bool pair = false;
    PairArgs pargs{};
    unsigned pair_threads = 0, pair_blocks = 0;
    size_t pair_lds = 0;
    bool pair_lt = false;
    unsigned* numts_alt = nullptr;
    unsigned pair_launches = 0;
    int pml_mode = kNoPml;
    unsigned n_unique_pml = 0;
    // Mur faces in creation order
    std::vector<MurDev> mur;
    // Mur face geometry (normal axis, face line, neighbour line), creation order
    struct MurGeo {
        int ny;
        unsigned line, shift;
    };
    std::vector<MurGeo> mur_geo;
    // quad sweep with Mur faces: sources on face / neighbour lines added after
    // the Mur hooks (exc_def[0]), the current update redone on the planes next
    // to each face (bands: axis, first and last plane) with the current sources
    // of those planes (exc_def[1])
    Exc exc_def[2];
    struct Band {
        int axis;
        unsigned lo, hi;
    };
    std::vector<Band> bands;
    // and at single cells: the currents reading a cell whose deferred source
    // changes it after the sweep, outside the bands (linear cell indices)
    unsigned long long* cell_list = nullptr;
    unsigned ncells = 0;
    std::vector<CurrAgain> curr_again;    // both, as the jobs of launches
    // lumped RLC and dispersive lists
    std::vector<RlcDev> rlc;
    std::vector<LorDev> lor;
    // their field elements and cells, and the steady-state probes' elements
    std::vector<std::vector<unsigned long long>> h_rlc;
    std::vector<std::vector<unsigned>> h_lor;
    std::vector<unsigned long long> h_ss;
    std::vector<int> lor_v, lor_i;
    // the extension hooks' launches (setup_hooks): before the voltage update,
    // after it (the steady-state evaluation follows launch hooks_ss), after
    // the current update
    std::vector<HookLaunch> hooks_pre, hooks_v, hooks_i;
    int hooks_ss = -1;
    bool pre_ahead = false;               // k_curr_pre can take hooks_pre of the next step

    // probes
    std::vector<ProbeDev> probes;
    std::vector<unsigned long long> h_elin;
    std::vector<signed char> h_esign;
    std::vector<double> h_ediv;
    ProbeDev* d_probes = nullptr;
    unsigned long long* d_elin = nullptr;
    signed char* d_esign = nullptr;
    double* d_ediv = nullptr;
    bool probes_dirty = false;
    unsigned min_interval = 0;

    // field dumps
    std::vector<DumpDev> dumps;
    std::vector<unsigned> dump_npts;
    bool sampled0 = false;          // the samples due before the first step were taken

    double* energy_part = nullptr;
    size_t read_rows = 0;           // x planes that read_buf holds
    float* read_buf = nullptr;      // of get_field; not in allocs, whose growth drops the captured chunks
    std::mutex read_mu;             // the read-out that uses it

    // steady-state detection
    bool has_ss = false;
    SteadyDev ss{};
    double* ss_part = nullptr;

    // timestep chunks replayed as HIP graphs: captured per launch pattern
    // (the probe / dump / steady-state decisions of the chunk's steps and the
    // buffer parity of the single-sweep forms), instantiated once, replayed
    struct GraphEnt {
        std::vector<unsigned char> key;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        size_t nalloc = 0;                // device allocations of the engine when captured
        unsigned pairs = 0;               // launches of k_pair in it
    };
    unsigned graph_chunk = 32;            // requested steps per graph (0: direct launches)
    unsigned graph_len = 0;               // steps per graph of the captured set
    std::vector<GraphEnt> graphs;
    unsigned graph_replays = 0, graph_captures = 0;

    // timing
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0, last_volt_ms = 0, last_curr_ms = 0;
    bool profile = false;
    std::vector<hipEvent_t> kev;

    template <typename T>
    int alloc(T** p, size_t n)
    {
        void* q = nullptr;
        const size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
        hipError_t e = device_malloc(this, &q, bytes);
        if (e != hipSuccess) return fail(EMS_E_NOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
        allocs.push_back(Alloc{q, bytes});
        alloc_bytes += bytes;
        *p = (T*)q;
        return 0;
    }
    bool drop_read_buf()
    {
        std::lock_guard<std::mutex> lk(read_mu);
        if (!read_buf) return false;
        (void)hipFree(read_buf);
        alloc_bytes -= read_rows * N[1] * N[2] * sizeof(float);
        read_buf = nullptr;
        return true;
    }
    void release(size_t k)
    {
        (void)hipFree(allocs[k].p);
        alloc_bytes -= allocs[k].bytes;
        allocs.erase(allocs.begin() + (std::ptrdiff_t)k);
    }
    unsigned long long lin(unsigned x, unsigned y, unsigned z) const
    {
        return x + (unsigned long long)N[0] * (y + (unsigned long long)N[1] * z);
    }
};

namespace {

void parallel_rows(size_t n, const std::function<void(size_t, size_t)>& fn)
{
    unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    if (n < 64 || nt == 1) {
        fn(0, n);
        return;
    }
    std::vector<std::thread> th;
    size_t per = (n + nt - 1) / nt;
    for (unsigned t = 0; t < nt; ++t) {
        size_t a = t * per, b = std::min(n, a + per);
        if (a >= b) break;
        th.emplace_back(fn, a, b);
    }
    for (auto& t : th) t.join();
}

// N-I-J-K host array -> device SoA (x fastest) staging buffer
void nijk_to_soa(const float* src, float* dst, const unsigned* N, unsigned long long cs)
{
    const size_t rows = (size_t)3 * N[1] * N[2];
    parallel_rows(rows, [&](size_t a, size_t b) {
        for (size_t r = a; r < b; ++r) {
            const unsigned n = (unsigned)(r / ((size_t)N[1] * N[2]));
            const size_t yz = r % ((size_t)N[1] * N[2]);
            const unsigned z = (unsigned)(yz / N[1]), y = (unsigned)(yz % N[1]);
            float* d = dst + n * cs + (size_t)N[0] * (y + (size_t)N[1] * z);
            for (unsigned x = 0; x < N[0]; ++x) d[x] = src[(((size_t)n * N[0] + x) * N[1] + y) * N[2] + z];
        }
    });
}

int upload_nijk(ems_engine* h, float* dptr, const float* host)
{
    std::vector<float> stage(3 * h->cs, 0.0f);
    nijk_to_soa(host, stage.data(), h->N, h->cs);
    HIPCHK(hipMemcpy(dptr, stage.data(), stage.size() * sizeof(float), hipMemcpyHostToDevice));
    return 0;
}

template <typename T>
int upload(ems_engine* h, T** d, const T* src, size_t n)
{
    int rc = h->alloc(d, n);
    if (rc) return rc;
    if (n) HIPCHK(hipMemcpy(*d, src, n * sizeof(T), hipMemcpyHostToDevice));
    return 0;
}

unsigned choose_zdepth(const unsigned* N)
{
    // z-sweep depth: 4 planes per thread measured best on MI355X (256^3 UPML:
    // 3 and 6 within 1 %, 8: +1.4 %, 16: +5 %, 32: +14 % step time; 1024 x
    // 1024 x 768 Mur: 8 +0.4 %); shallower sweeps when the grid would
    // otherwise give fewer than 2048 workgroups for 256 CUs
    const unsigned plane = N[0] * N[1];
    const unsigned qt = (plane + kBlock - 1) / kBlock;
    unsigned d = 4;
    while (d > 1 && (unsigned long long)qt * ((N[2] + d - 1) / d) < 2048ull) d /= 2;
    return d;
}

}  // namespace

namespace {

// per-device address of `scratch`, taken once per device with that device
// current (each device holds its own copy of the array at its own address)
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

int scratch_setup(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (device < 0 || device >= kMaxDevices) return fail(EMS_E_ARG, "device ordinal beyond the scratch table");
    if (g_scratch_ptr[device]) return 0;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return fail(EMS_E_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_ptr[device] = static_cast<double*>(p);
    return 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

const char* ems_last_error(void) { return g_err.c_str(); }

int ems_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int ems_create_layout(ems_engine** out, const unsigned numLines[3], const float* vv, const float* vi,
                      const float* ii, const float* iv, int device, int layout)
{
    if (!out || !numLines || !vv || !vi || !ii || !iv) return fail(EMS_E_ARG, "null argument");
    *out = nullptr;
    if (layout < EMS_LAYOUT_AUTO || layout > EMS_LAYOUT_COMPRESSED) return fail(EMS_E_ARG, "unknown layout");
    for (int n = 0; n < 3; ++n)
        if (numLines[n] < 3) return fail(EMS_E_ARG, "at least 3 mesh lines per direction are required");
    const unsigned long long plane = (unsigned long long)numLines[0] * numLines[1];
    if (plane > 0xFFFFFFFFull || plane * numLines[2] > 0xFFFFFFFFull)
        return fail(EMS_E_ARG, "mesh too large for 32-bit in-plane indexing");
    int ndev = ems_device_count();
    if (ndev <= 0) return fail(EMS_E_NODEV, "no HIP device available");
    if (device < 0 || device >= ndev) return fail(EMS_E_ARG, "invalid device ordinal");
    HIPCHK(hipSetDevice(device));
    if (int src = scratch_setup(device)) return src;
    const unsigned long long tot = plane * numLines[2];
    const unsigned long long cs = (tot + 63) / 64 * 64;
    // per-cell compression (host): first-seen order x -> y -> z
    std::vector<uint16_t> cidx;
    std::vector<float> tab[2];
    size_t U = 0;
    if (layout != EMS_LAYOUT_PLAIN) {
        U = ems::compress_cells(numLines, vv, vi, ii, iv, cs, cidx, tab[0], tab[1], ems::host_threads());
        if (U == 0 && layout == EMS_LAYOUT_COMPRESSED)
            return fail(EMS_E_ARG, "the operator has more than 65536 unique coefficient tuples");
        if (layout == EMS_LAYOUT_AUTO && U * 16 > tot) U = 0;
    }
    ems_engine* h = new ems_engine();
    h->device = device;
    h->layout_req = layout;
    for (int n = 0; n < 3; ++n) h->N[n] = numLines[n];
    h->cs = cs;
    GridDesc& g = h->g;
    g.Nx = numLines[0];
    g.Ny = numLines[1];
    g.Nz = numLines[2];
    g.plane = (unsigned)plane;
    g.cs = h->cs;
    g.zdepth = choose_zdepth(h->N);
    if (const char* zd = std::getenv("EMS_ZDEPTH")) {
        const int v = std::atoi(zd);
        if (v >= 1 && v <= 1024) g.zdepth = (unsigned)v;
    }
    set_tiles(g, 0);
    // fields larger than the last-level cache (256 MB on MI355X) stream through it
    h->nt_fields = 2ull * 3ull * h->cs * sizeof(float) > (192ull << 20);
    if (const char* nt = std::getenv("EMS_NT_FIELDS")) h->nt_fields = std::atoi(nt) != 0;
    if (const char* db = std::getenv("EMS_DEVICE_BYTES")) h->alloc_most = (size_t)std::strtoull(db, nullptr, 10);
    if (const char* qe = std::getenv("EMS_QUAD")) h->quad_req = std::atoi(qe) ? -1 : 0;
    if (const char* gc = std::getenv("EMS_GRAPH_CHUNK")) {
        const int v = std::atoi(gc);
        if (v >= 0 && v <= 1 << 20) h->graph_chunk = (unsigned)v;
    }
    int rc = 0;
    auto bail = [&](int r) {
        ems_destroy(h);
        return r;
    };
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) return bail(fail(EMS_E_HIP, "stream creation failed"));
    if ((rc = h->alloc(&h->V, 3 * h->cs)) || (rc = h->alloc(&h->I, 3 * h->cs)) || (rc = h->alloc(&h->numts_dev, 4)))
        return bail(rc);
    if (hipMemset(h->V, 0, 3 * h->cs * sizeof(float)) != hipSuccess ||
        hipMemset(h->I, 0, 3 * h->cs * sizeof(float)) != hipSuccess ||
        hipMemset(h->numts_dev, 0, 4 * sizeof(unsigned)) != hipSuccess)
        return bail(fail(EMS_E_HIP, "hipMemset failed"));
    if (U > 0) {
        h->cmp = true;
        h->n_unique = (unsigned)U;
        if ((rc = upload(h, &h->cidx, (const unsigned short*)cidx.data(), cidx.size())) ||
            (rc = upload(h, &h->ctab[0], tab[0].data(), tab[0].size())) ||
            (rc = upload(h, &h->ctab[1], tab[1].data(), tab[1].size())))
            return bail(rc);
    } else {
        if ((rc = h->alloc(&h->vv, 3 * h->cs)) || (rc = h->alloc(&h->vi, 3 * h->cs)) ||
            (rc = h->alloc(&h->ii, 3 * h->cs)) || (rc = h->alloc(&h->iv, 3 * h->cs)))
            return bail(rc);
        if ((rc = upload_nijk(h, h->vv, vv)) || (rc = upload_nijk(h, h->vi, vi)) || (rc = upload_nijk(h, h->ii, ii)) ||
            (rc = upload_nijk(h, h->iv, iv)))
            return bail(rc);
    }
    h->kV = CoefArgs{h->vv, h->vi, h->cidx, (const float4*)h->ctab[0], 2u * h->n_unique};
    h->kI = CoefArgs{h->ii, h->iv, h->cidx, (const float4*)h->ctab[1], 2u * h->n_unique};
    hipEventCreate(&h->ev0);
    hipEventCreate(&h->ev1);
    *out = h;
    return 0;
}

int ems_create(ems_engine** out, const unsigned numLines[3], const float* vv, const float* vi, const float* ii,
               const float* iv, int device)
{
    return ems_create_layout(out, numLines, vv, vi, ii, iv, device, EMS_LAYOUT_AUTO);
}

int ems_create_sse_compressed(ems_engine** out, const unsigned numLines[3], const unsigned* op_index,
                              unsigned n_unique, const float* const vv4[3], const float* const vi4[3],
                              const float* const ii4[3], const float* const iv4[3], int device, int layout)
{
    if (!out || !numLines) return fail(EMS_E_ARG, "null argument");
    *out = nullptr;
    const size_t M = (size_t)numLines[0] * numLines[1] * numLines[2];
    std::vector<float> a(3 * M), b(3 * M), c(3 * M), d(3 * M);
    const int rc = ems_expand_sse_compressed(numLines, op_index, n_unique, vv4, vi4, ii4, iv4, a.data(), b.data(),
                                             c.data(), d.data());
    if (rc) return rc;
    return ems_create_layout(out, numLines, a.data(), b.data(), c.data(), d.data(), device, layout);
}

int ems_compress_operator(const unsigned numLines[3], const float* vv, const float* vi, const float* ii,
                          const float* iv, unsigned short* idx, float* tabV, float* tabI, unsigned max_unique)
{
    if (!numLines || !vv || !vi || !ii || !iv || !idx || !tabV || !tabI) return fail(EMS_E_ARG, "null argument");
    const unsigned long long tot = (unsigned long long)numLines[0] * numLines[1] * numLines[2];
    if (tot == 0) return fail(EMS_E_ARG, "empty mesh");
    std::vector<uint16_t> ci;
    std::vector<float> tv, ti;
    const size_t U = ems::compress_cells(numLines, vv, vi, ii, iv, tot, ci, tv, ti, ems::host_threads());
    if (U == 0 || U > max_unique) return fail(EMS_E_ARG, "more unique coefficient tuples than the table holds");
    std::memcpy(idx, ci.data(), tot * sizeof(uint16_t));
    std::memcpy(tabV, tv.data(), tv.size() * sizeof(float));
    std::memcpy(tabI, ti.data(), ti.size() * sizeof(float));
    return (int)U;
}

int ems_expand_sse_compressed(const unsigned numLines[3], const unsigned* op_index, unsigned n_unique,
                              const float* const vv4[3], const float* const vi4[3], const float* const ii4[3],
                              const float* const iv4[3], float* vv, float* vi, float* ii, float* iv)
{
    if (!numLines || !op_index || !vv4 || !vi4 || !ii4 || !iv4 || !vv || !vi || !ii || !iv)
        return fail(EMS_E_ARG, "null argument");
    for (int n = 0; n < 3; ++n)
        if (!vv4[n] || !vi4[n] || !ii4[n] || !iv4[n]) return fail(EMS_E_ARG, "null compressed table");
    if (n_unique == 0) return fail(EMS_E_ARG, "empty compressed table");
    const size_t Nx = numLines[0], Ny = numLines[1], Nz = numLines[2], nV = (Nz + 3) / 4;
    for (size_t xy = 0; xy < Nx * Ny; ++xy)
        for (size_t v = 0; v < nV; ++v)
            if (op_index[xy * Nz + v] >= n_unique) return fail(EMS_E_ARG, "compressed index outside the table");
    ems::expand_sse_compressed(numLines, op_index, n_unique, vv4, vi4, ii4, iv4, vv, vi, ii, iv, ems::host_threads());
    return 0;
}

int ems_get_layout(const ems_engine* h, int* layout, unsigned* n_unique, int* pml_layout, unsigned* n_unique_pml)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (layout) *layout = h->cmp ? EMS_LAYOUT_COMPRESSED : EMS_LAYOUT_PLAIN;
    if (n_unique) *n_unique = h->n_unique;
    if (pml_layout)
        *pml_layout = h->pml_mode == kPmlCompressed ? EMS_LAYOUT_COMPRESSED
                      : h->pml_mode == kPmlPlain    ? EMS_LAYOUT_PLAIN
                                                    : 0;
    if (n_unique_pml) *n_unique_pml = h->n_unique_pml;
    return 0;
}

}  // extern "C"

// entries (list order) grouped per (component, cell) in order of first
// appearance, as the Excite hook applies them, uploaded into E (device lists only)
static int upload_exc_groups(ems_engine* h, const std::vector<ExcEnt>& ent, ems_engine::Exc& E)
{
    const unsigned K = (unsigned)ent.size();
    E.K = K;
    E.G = 0;
    if (!K) return 0;
    std::unordered_map<unsigned long long, unsigned> gid;
    std::vector<unsigned long long> glin;
    std::vector<unsigned> grp(K);
    for (unsigned k = 0; k < K; ++k) {
        const unsigned long long l = ent[k].dir * h->cs + h->lin(ent[k].x, ent[k].y, ent[k].z);
        auto it = gid.find(l);
        if (it == gid.end()) {
            it = gid.emplace(l, (unsigned)glin.size()).first;
            glin.push_back(l);
        }
        grp[k] = it->second;
    }
    const unsigned G = (unsigned)glin.size();
    std::vector<unsigned> gbeg(G + 1, 0), order(K);
    for (unsigned k = 0; k < K; ++k) ++gbeg[grp[k] + 1];
    for (unsigned g = 0; g < G; ++g) gbeg[g + 1] += gbeg[g];
    std::vector<unsigned> fill(gbeg.begin(), gbeg.end() - 1);
    for (unsigned k = 0; k < K; ++k) order[fill[grp[k]]++] = k;
    std::vector<float> ga(K);
    std::vector<unsigned> gd(K);
    for (unsigned k = 0; k < K; ++k) {
        ga[k] = ent[order[k]].amp;
        gd[k] = ent[order[k]].delay;
    }
    E.G = G;
    E.h_glin = glin;
    int rc;
    if ((rc = upload(h, &E.gbeg, gbeg.data(), G + 1)) || (rc = upload(h, &E.glin, glin.data(), G)) ||
        (rc = upload(h, &E.amp, ga.data(), K)) || (rc = upload(h, &E.delay, gd.data(), K)))
        return rc;
    return 0;
}

extern "C" {

int ems_set_excitation(ems_engine* h, const float* sig_volt, const float* sig_curr, unsigned length, int period_steps,
                       unsigned nvolt, const unsigned* vidx, const unsigned short* vdir, const float* vamp,
                       const unsigned* vdelay, unsigned ncurr, const unsigned* cidx, const unsigned short* cdir,
                       const float* camp, const unsigned* cdelay)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (h->has_exc) return fail(EMS_E_STATE, "excitation already set");
    if (length == 0 || !sig_volt || !sig_curr) return fail(EMS_E_ARG, "empty excitation signal");
    HIPCHK(hipSetDevice(h->device));
    int rc;
    if ((rc = upload(h, &h->sig[0], sig_volt, length)) || (rc = upload(h, &h->sig[1], sig_curr, length))) return rc;
    h->sigLen = length;
    h->period = period_steps;
    const unsigned Ks[2] = {nvolt, ncurr};
    const unsigned* idx[2] = {vidx, cidx};
    const unsigned short* dir[2] = {vdir, cdir};
    const float* amp[2] = {vamp, camp};
    const unsigned* del[2] = {vdelay, cdelay};
    for (int c = 0; c < 2; ++c) {
        const unsigned K = Ks[c];
        auto& E = h->exc[c];
        E.K = K;
        if (!K) continue;
        if (!idx[c] || !dir[c] || !amp[c] || !del[c]) return fail(EMS_E_ARG, "null excitation list");
        // group the entries by (component, cell) in order of first appearance
        std::unordered_map<unsigned long long, unsigned> gid;
        std::vector<unsigned long long> glin;
        std::vector<unsigned> grp(K);
        E.host.resize(K);
        for (unsigned k = 0; k < K; ++k) {
            const unsigned x = idx[c][k], y = idx[c][K + k], z = idx[c][2 * K + k];
            if (x >= h->N[0] || y >= h->N[1] || z >= h->N[2] || dir[c][k] > 2)
                return fail(EMS_E_ARG, "excitation cell outside the mesh");
            const unsigned long long l = dir[c][k] * h->cs + h->lin(x, y, z);
            auto it = gid.find(l);
            if (it == gid.end()) {
                it = gid.emplace(l, (unsigned)glin.size()).first;
                glin.push_back(l);
            }
            grp[k] = it->second;
            E.host[k] = ExcEnt{(unsigned short)std::min(x, 65535u), (unsigned short)std::min(y, 65535u),
                               (unsigned short)std::min(z, 65535u), dir[c][k], amp[c][k], del[c][k]};
        }
        const unsigned G = (unsigned)glin.size();
        std::vector<unsigned> gbeg(G + 1, 0), order(K);
        for (unsigned k = 0; k < K; ++k) ++gbeg[grp[k] + 1];
        for (unsigned g = 0; g < G; ++g) gbeg[g + 1] += gbeg[g];
        std::vector<unsigned> fill(gbeg.begin(), gbeg.end() - 1);
        for (unsigned k = 0; k < K; ++k) order[fill[grp[k]]++] = k;   // stable: list order inside a group
        std::vector<float> ga(K);
        std::vector<unsigned> gd(K);
        for (unsigned k = 0; k < K; ++k) {
            ga[k] = amp[c][order[k]];
            gd[k] = del[c][order[k]];
        }
        E.G = G;
        E.h_gbeg = gbeg;
        E.h_glin = glin;
        E.h_amp = ga;
        E.h_delay = gd;
        if ((rc = upload(h, &E.gbeg, gbeg.data(), G + 1)) || (rc = upload(h, &E.glin, glin.data(), G)) ||
            (rc = upload(h, &E.amp, ga.data(), K)) || (rc = upload(h, &E.delay, gd.data(), K)))
            return rc;
    }
    h->has_exc = true;
    return 0;
}

int ems_add_upml(ems_engine* h, const unsigned start[3], const unsigned num[3], const float* vv, const float* vvfo,
                 const float* vvfn, const float* ii, const float* iifo, const float* iifn)
{
    if (!h || !start || !num || !vv || !vvfo || !vvfn || !ii || !iifo || !iifn) return fail(EMS_E_ARG, "null argument");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (h->slabs.size() >= kMaxSlabs) return fail(EMS_E_ARG, "at most 6 UPML slabs");
    for (int n = 0; n < 3; ++n)
        if (num[n] == 0 || start[n] + num[n] > h->N[n]) return fail(EMS_E_ARG, "UPML slab outside the mesh");
    SlabTab t{};
    t.x0 = start[0];
    t.y0 = start[1];
    t.z0 = start[2];
    t.x1 = start[0] + num[0] - 1;
    t.y1 = start[1] + num[1] - 1;
    t.z1 = start[2] + num[2] - 1;
    t.xo = (int)(start[0] & ~3u);
    t.nx = ((start[0] + num[0] + 3u) & ~3u) - (unsigned)t.xo;
    t.ny = num[1];
    for (const auto& o : h->slabs) {
        const SlabTab& u = o.tab;
        const bool overlap = t.x0 <= u.x1 && t.x1 >= u.x0 && t.y0 <= u.y1 && t.y1 >= u.y0 && t.z0 <= u.z1 && t.z1 >= u.z0;
        if (overlap) return fail(EMS_E_ARG, "overlapping UPML slabs are not supported");
    }
    ems_engine::SlabHost sh;
    sh.tab = t;
    sh.cnt = (unsigned long long)num[0] * num[1] * num[2];
    for (int n = 0; n < 3; ++n) sh.num[n] = num[n];
    // repack [3][nx][ny][nz] (z fastest) -> [3][nz][ny][nx] (x fastest)
    auto repack = [&](const float* src, std::vector<float>& d) {
        d.resize(3 * sh.cnt);
        for (int n = 0; n < 3; ++n)
            for (unsigned x = 0; x < num[0]; ++x)
                for (unsigned y = 0; y < num[1]; ++y)
                    for (unsigned z = 0; z < num[2]; ++z)
                        d[n * sh.cnt + x + (unsigned long long)num[0] * (y + (unsigned long long)num[1] * z)] =
                            src[(((size_t)n * num[0] + x) * num[1] + y) * num[2] + z];
    };
    repack(vv, sh.v[0]);
    repack(vvfo, sh.v[1]);
    repack(vvfn, sh.v[2]);
    repack(ii, sh.i[0]);
    repack(iifo, sh.i[1]);
    repack(iifn, sh.i[2]);
    h->slabs.push_back(std::move(sh));
    return 0;
}

static int upload_upml(ems_engine* h)
{
    // All slabs' positions are numbered consecutively, each slab from a
    // multiple of 4 and padded along x to whole groups of four cells
    // (SlabTab); every array is [k][npos], padding positions hold zeros.
    // Plain: coef[9][npos] per half step.  Compressed: one index array into
    // a table of the unique 18-float tuples (V: c0, cfo, cfn; I: likewise),
    // numbered in first-seen order over the cells slab after slab, x fastest
    // (padding positions take entry 0).
    if (h->slabs.empty()) return 0;
    unsigned long long npos = 0, ncell = 0;
    std::vector<unsigned long long> first;      // first cell of each slab (compact count)
    for (auto& s : h->slabs) {
        npos = (npos + 3) & ~3ull;
        s.tab.off = npos;
        npos += (unsigned long long)s.tab.nx * s.num[1] * s.num[2];
        first.push_back(ncell);
        ncell += s.cnt;
    }
    if (npos >= 0xFFFFFFFFull) return fail(EMS_E_ARG, "too many UPML positions for 32-bit numbering");
    // position of cell j (compact, x fastest) of slab k
    auto pos_of = [&](size_t k, unsigned long long j) {
        const auto& S = h->slabs[k];
        const unsigned long long xs = j % S.num[0], r = j / S.num[0];
        const unsigned long long ys = r % S.num[1], zs = r / S.num[1];
        return S.tab.off + (unsigned long long)(S.tab.x0 - S.tab.xo) + xs + S.tab.nx * (ys + (unsigned long long)S.tab.ny * zs);
    };
    std::vector<uint32_t> pidx;
    std::vector<float> uniq;
    size_t U = 0;
    if (h->layout_req != EMS_LAYOUT_PLAIN) {
        auto get = [&](size_t i, float* t) {
            size_t s = 0;
            while (s + 1 < first.size() && i >= first[s + 1]) ++s;
            const auto& S = h->slabs[s];
            const unsigned long long j = i - first[s], cnt = S.cnt;
            for (int a = 0; a < 3; ++a)
                for (int n = 0; n < 3; ++n) {
                    t[3 * a + n] = S.v[a][n * cnt + j];
                    t[9 + 3 * a + n] = S.i[a][n * cnt + j];
                }
        };
        U = ems::dedup_tuples<18>(ncell, get, pidx, uniq, 65536, ems::host_threads());
        if (h->layout_req == EMS_LAYOUT_AUTO && U * 16 > ncell) U = 0;
    }
    const bool cmp = U > 0;
    int rc;
    unsigned* dpidx = nullptr;
    if (cmp) {
        std::vector<uint32_t> ppos(npos, 0u);
        for (size_t k = 0; k < h->slabs.size(); ++k)
            for (unsigned long long j = 0; j < h->slabs[k].cnt; ++j) ppos[pos_of(k, j)] = pidx[first[k] + j];
        if ((rc = upload(h, &dpidx, ppos.data(), ppos.size()))) return rc;
    }
    for (int side = 0; side < 2; ++side) {
        PmlArgs& P = side ? h->pmlI : h->pmlV;
        P = PmlArgs{};
        P.n = (int)h->slabs.size();
        P.npos = npos;
        for (size_t k = 0; k < h->slabs.size(); ++k) P.tab[k] = h->slabs[k].tab;
        if (cmp) {
            std::vector<float> pt(U * 12, 0.0f);
            for (size_t u = 0; u < U; ++u)
                for (int q = 0; q < 9; ++q) pt[u * 12 + q] = uniq[u * 18 + 9 * side + q];
            float* dpt;
            if ((rc = upload(h, &dpt, pt.data(), pt.size()))) return rc;
            P.ptab = (const float4*)dpt;
            P.pidx = dpidx;
        } else {
            std::vector<float> stage(9 * npos, 0.0f);
            for (size_t k = 0; k < h->slabs.size(); ++k) {
                const auto& S = h->slabs[k];
                const auto* src = side ? S.i : S.v;
                for (unsigned long long j = 0; j < S.cnt; ++j) {
                    const unsigned long long q = pos_of(k, j);
                    for (int a = 0; a < 3; ++a)
                        for (int n = 0; n < 3; ++n) stage[(3 * a + n) * npos + q] = src[a][n * S.cnt + j];
                }
            }
            float* dc;
            if ((rc = upload(h, &dc, stage.data(), stage.size()))) return rc;
            P.coef = dc;
        }
        float* fl;
        if ((rc = h->alloc(&fl, 3 * npos))) return rc;
        HIPCHK(hipMemset(fl, 0, 3 * npos * sizeof(float)));
        P.flux_in = fl;
        P.flux_out = fl;
    }
    h->pml_mode = cmp ? kPmlCompressed : kPmlPlain;
    h->n_unique_pml = cmp ? (unsigned)U : 0;
    h->slabs.clear();
    return 0;
}

int ems_add_mur(ems_engine* h, int ny, unsigned line, unsigned line_shift, const float* coeff_nyP,
                const float* coeff_nyPP, unsigned start_ts)
{
    if (!h || !coeff_nyP || !coeff_nyPP) return fail(EMS_E_ARG, "null argument");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (ny < 0 || ny > 2 || line >= h->N[ny] || line_shift >= h->N[ny]) return fail(EMS_E_ARG, "bad Mur face");
    HIPCHK(hipSetDevice(h->device));
    const int nyP = (ny + 1) % 3, nyPP = (ny + 2) % 3;
    MurDev m{};
    m.na = h->N[nyP];
    m.nb = h->N[nyPP];
    m.offP = nyP * h->cs;
    m.offPP = nyPP * h->cs;
    m.start_ts = start_ts;
    const size_t cnt = (size_t)m.na * m.nb;
    // device order of the face points: the lower tangential axis fastest (x
    // for y and z faces, y for x faces), so that neighbouring threads touch
    // neighbouring field elements; the caller's arrays are [nyP][nyPP]
    const bool tr = nyP < nyPP;
    std::vector<unsigned> face(cnt), shift(cnt);
    std::vector<float> cP(cnt), cPP(cnt);
    for (unsigned i = 0; i < m.na; ++i)
        for (unsigned j = 0; j < m.nb; ++j) {
            unsigned p[3], s[3];
            p[ny] = line;
            s[ny] = line_shift;
            p[nyP] = s[nyP] = i;
            p[nyPP] = s[nyPP] = j;
            const size_t src = (size_t)i * m.nb + j, k = tr ? (size_t)j * m.na + i : src;
            face[k] = (unsigned)h->lin(p[0], p[1], p[2]);
            shift[k] = (unsigned)h->lin(s[0], s[1], s[2]);
            cP[k] = coeff_nyP[src];
            cPP[k] = coeff_nyPP[src];
        }
    int rc;
    unsigned *df, *dsh;
    float *dcp, *dcpp;
    if ((rc = upload(h, &df, face.data(), cnt)) || (rc = upload(h, &dsh, shift.data(), cnt)) ||
        (rc = upload(h, &dcp, cP.data(), cnt)) || (rc = upload(h, &dcpp, cPP.data(), cnt)) ||
        (rc = h->alloc(&m.mP, cnt)) || (rc = h->alloc(&m.mPP, cnt)))
        return rc;
    HIPCHK(hipMemset(m.mP, 0, cnt * sizeof(float)));
    HIPCHK(hipMemset(m.mPP, 0, cnt * sizeof(float)));
    m.face = df;
    m.shift = dsh;
    m.cP = dcp;
    m.cPP = dcpp;
    h->mur.push_back(m);
    h->mur_geo.push_back(ems_engine::MurGeo{ny, line, line_shift});
    return 0;
}

int ems_add_lumped_rlc(ems_engine* h, unsigned count, const unsigned* pos, const int* dir, const float* const coeffs[9])
{
    if (!h || !pos || !dir || !coeffs) return fail(EMS_E_ARG, "null argument");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (!count) return 0;
    HIPCHK(hipSetDevice(h->device));
    RlcDev r{};
    r.count = count;
    std::vector<unsigned long long> lin(count);
    for (unsigned k = 0; k < count; ++k) {
        const unsigned x = pos[k], y = pos[count + k], z = pos[2 * count + k];
        if (x >= h->N[0] || y >= h->N[1] || z >= h->N[2] || dir[k] < 0 || dir[k] > 2)
            return fail(EMS_E_ARG, "lumped element outside the mesh");
        lin[k] = dir[k] * h->cs + h->lin(x, y, z);
    }
    int rc;
    unsigned long long* dl;
    if ((rc = upload(h, &dl, lin.data(), count))) return rc;
    r.lin = dl;
    for (int c = 0; c < 9; ++c) {
        float* d;
        if (!coeffs[c]) return fail(EMS_E_ARG, "null RLC coefficient array");
        if ((rc = upload(h, &d, coeffs[c], count))) return rc;
        r.c[c] = d;
    }
    if ((rc = h->alloc(&r.vd, 3 * count)) || (rc = h->alloc(&r.jn, 3 * count)) || (rc = h->alloc(&r.il, count)))
        return rc;
    HIPCHK(hipMemset(r.vd, 0, 3 * count * sizeof(float)));
    HIPCHK(hipMemset(r.jn, 0, 3 * count * sizeof(float)));
    HIPCHK(hipMemset(r.il, 0, count * sizeof(float)));
    h->rlc.push_back(r);
    h->h_rlc.push_back(std::move(lin));
    return 0;
}

int ems_add_lorentz(ems_engine* h, unsigned count, const unsigned* pos, const float* v_int, const float* v_ext,
                    const float* v_lor, const float* i_int, const float* i_ext, const float* i_lor, int volt_on,
                    int curr_on)
{
    if (!h || !pos) return fail(EMS_E_ARG, "null argument");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (!count) return 0;
    HIPCHK(hipSetDevice(h->device));
    std::vector<unsigned> lin(count);
    for (unsigned k = 0; k < count; ++k) {
        const unsigned x = pos[k], y = pos[count + k], z = pos[2 * count + k];
        if (x >= h->N[0] || y >= h->N[1] || z >= h->N[2]) return fail(EMS_E_ARG, "dispersive cell outside the mesh");
        lin[k] = (unsigned)h->lin(x, y, z);
    }
    int rc;
    unsigned* dl;
    if ((rc = upload(h, &dl, lin.data(), count))) return rc;
    for (int side = 0; side < 2; ++side) {
        const bool on = side ? curr_on : volt_on;
        LorDev d{};
        d.count = count;
        d.lin = dl;
        const float* ci = side ? i_int : v_int;
        const float* ce = side ? i_ext : v_ext;
        const float* cl = side ? i_lor : v_lor;
        if (on) {
            if (!ci || !ce) return fail(EMS_E_ARG, "null ADE coefficient array");
            float *a, *b, *c = nullptr;
            if ((rc = upload(h, &a, ci, 3 * count)) || (rc = upload(h, &b, ce, 3 * count))) return rc;
            if (cl && (rc = upload(h, &c, cl, 3 * count))) return rc;
            d.cint = a;
            d.cext = b;
            d.clor = c;
            if ((rc = h->alloc(&d.ade, 3 * count)) || (rc = h->alloc(&d.lor, 3 * count))) return rc;
            HIPCHK(hipMemset(d.ade, 0, 3 * count * sizeof(float)));
            HIPCHK(hipMemset(d.lor, 0, 3 * count * sizeof(float)));
        }
        h->lor.push_back(d);
        (side ? h->lor_i : h->lor_v).push_back(on ? 1 : 0);
    }
    h->h_lor.push_back(std::move(lin));
    return 0;
}

// z-sweep depth of the fused step: 16 planes per workgroup, shallower when
// the grid would otherwise give fewer than 1024 workgroups
static unsigned choose_fused_zdepth(unsigned ntiles, unsigned Nz)
{
    unsigned d = 16;
    while (d > 4 && (unsigned long long)ntiles * ((Nz + d - 1) / d) < 1024ull) d /= 2;
    if (const char* zd = std::getenv("EMS_FZDEPTH")) {
        const int v = std::atoi(zd);
        if (v >= 1 && v <= 1024) d = (unsigned)v;
    }
    return d;
}

// Decide and prepare the fused single-sweep step: every active extension
// must have a fused form (UPML, excitation); Mur, Lorentz and lumped RLC keep
// the two-half-step path.  Form 1 (k_step) stages V^{n+1} planes in LDS per
// 64 x 16 tile; form 2 (k_step2) sweeps single columns and recomputes the
// neighbour components it needs.
static int setup_fused(ems_engine* h)
{
    h->fused = 0;
    // automatic mode: the tiled quad sweep (form 3, k_step4t) on meshes
    // without UPML whose rows hold at least 64 quads (1024 x 1024 x 768 Mur
    // layers 12.08 -> 11.65 ms per step, 256^3 PEC 0.218 -> 0.202 ms), where
    // every extension has a form for it; two half steps elsewhere (256^3
    // UPML, compressed: 0.50 ms per step in the LDS sweep, 0.38 ms in two
    // half steps)
    int form = h->fused_req;
    const bool autom = form == -1;
    if (autom) {
        bool sweep = !h->pmlV.n && h->quad_req != 0 && h->N[0] % 4 == 0 && h->N[0] / 4 >= 64;
        if (const char* as = std::getenv("EMS_AUTO_SWEEP")) sweep = sweep && std::atoi(as) != 0;
        if (sweep) {
            // the sweep keeps a second copy of both fields: only where it fits
            // with 1 GiB to spare
            size_t freeb = 0, totalb = 0;
            const size_t need = 6 * h->cs * sizeof(float) + (1ull << 30);
            if (hipMemGetInfo(&freeb, &totalb) != hipSuccess || freeb < need) sweep = false;
        }
        if (!sweep) return 0;
        form = 3;
    }
    if (form <= 0) return 0;
    std::string why;
    const unsigned Nx = h->N[0], Ny = h->N[1], Nz = h->N[2];
    if (!h->mur.empty() && form != 3) why = "Mur ABC has no fused form but the quad sweep's";
    else if (!h->lor.empty()) why = "Lorentz / Drude materials have no fused form";
    else if (!h->rlc.empty()) why = "lumped RLC elements have no fused form";
    else if (h->has_ss) why = "steady-state detection has no fused form";
    else if (Nx >= 65535 || Ny >= 65535 || Nz >= 65535) why = "mesh too large for the fused step";
    for (const auto& e : h->exc[1].host)
        if (why.empty() && (e.x + 1u >= Nx || e.y + 1u >= Ny || e.z + 1u >= Nz))
            why = "a current source lies outside the updated range";
    // source lists in list order: per tile (form 1: voltage sources of the
    // tile and its halo, column x0+kTX and row y0+kTY; current sources of the
    // tile) or per (x, y) column (form 2)
    const unsigned ntx = (Nx + kTX - 1) / kTX, nty = (Ny + kTY - 1) / kTY;
    if (why.empty() && form == 3) {
        if (h->pmlV.n) why = "the quad sweep has no UPML form";
        else if (Nx % 4) why = "the quad sweep needs a multiple of 4 x lines";
    }
    // quad sweep with Mur faces: voltage sources on a face or neighbour line
    // wait for the Mur hooks (exc_def[0]); the current update of the planes
    // whose voltages the hooks and those sources change is redone (bands)
    std::vector<ExcEnt> deferred[2];
    auto on_face = [&](const ExcEnt& e) {
        const unsigned p[3] = {e.x, e.y, e.z};
        for (const auto& f : h->mur_geo)
            if (p[f.ny] == f.line || p[f.ny] == f.shift) return true;
        return false;
    };
    h->bands.clear();
    h->ncells = 0;
    h->mur_fold[0] = h->mur_fold[1] = -1;
    std::vector<unsigned long long> cells;
    if (why.empty() && form == 3) {
        // k_step4t on rows of at least 64 quads (EMS_Q4TILE forces it on or off)
        h->q4tile = Nx / 4 >= 64;
        if (const char* te = std::getenv("EMS_Q4TILE")) h->q4tile = std::atoi(te) != 0;
        // it runs the pre and post hooks of the Mur faces on x = 0 and
        // x = Nx-1 and updates the currents next to them itself
        bool fold = h->q4tile && Nx >= 8;
        if (const char* mf = std::getenv("EMS_MUR_FOLD")) fold = fold && std::atoi(mf) != 0;
        for (size_t k = 0; k < h->mur_geo.size() && fold; ++k) {
            const auto& f = h->mur_geo[k];
            if (f.ny != 0) continue;
            if (f.line == 0 && f.shift == 1 && h->mur_fold[0] < 0) h->mur_fold[0] = (int)k;
            else if (f.line == Nx - 1 && f.shift == Nx - 2 && h->mur_fold[1] < 0) h->mur_fold[1] = (int)k;
        }
        // the Mur apply sets the voltages of the face line only; the current
        // at plane k reads the voltages of planes k and k+1 along the normal
        for (size_t k = 0; k < h->mur_geo.size(); ++k) {
            const auto& f = h->mur_geo[k];
            if ((int)k == h->mur_fold[0] || (int)k == h->mur_fold[1]) continue;
            const unsigned lo = f.line ? f.line - 1 : 0, hi = std::min(f.line, h->N[f.ny] - 2);
            if (lo <= hi) h->bands.push_back(ems_engine::Band{f.ny, lo, hi});
        }
        auto in_band = [&](const unsigned p[3]) {
            for (const auto& b : h->bands)
                if (p[b.axis] >= b.lo && p[b.axis] <= b.hi) return true;
            return false;
        };
        // a deferred voltage source changes its cell after the sweep: the
        // currents of the cell and of its -x, -y, -z neighbours read it
        for (const auto& e : h->exc[0].host) {
            if (!on_face(e)) continue;
            for (int d = 0; d < 4; ++d) {
                unsigned p[3] = {e.x, e.y, e.z};
                if (d < 3) {
                    if (!p[d]) continue;
                    --p[d];
                }
                if (p[0] + 1 >= Nx || p[1] + 1 >= Ny || p[2] + 1 >= Nz || in_band(p)) continue;
                cells.push_back(h->lin(p[0], p[1], p[2]));
            }
        }
        std::sort(cells.begin(), cells.end());
        cells.erase(std::unique(cells.begin(), cells.end()), cells.end());
        for (const auto& e : h->exc[1].host) {
            const unsigned p[3] = {e.x, e.y, e.z};
            if (in_band(p) || std::binary_search(cells.begin(), cells.end(), h->lin(e.x, e.y, e.z)))
                deferred[1].push_back(e);
        }
    }
    const unsigned nlists = form == 1 ? ntx * nty : h->g.plane;
    std::vector<std::vector<ExcEnt>> lists[2];
    size_t most = 0;
    for (int c = 0; c < 2 && why.empty(); ++c) {
        lists[c].assign(nlists, {});
        for (const auto& e : h->exc[c].host) {
            if (form == 3 && c == 0 && !h->mur_geo.empty() && on_face(e)) {
                deferred[0].push_back(e);
                continue;
            }
            if (form >= 2) {
                lists[c][e.x + Nx * (unsigned)e.y].push_back(e);
                continue;
            }
            const unsigned txs[2] = {e.x / kTX, (c == 0 && e.x % kTX == 0 && e.x > 0) ? e.x / kTX - 1 : ~0u};
            const unsigned tys[2] = {e.y / kTY, (c == 0 && e.y % kTY == 0 && e.y > 0) ? e.y / kTY - 1 : ~0u};
            for (unsigned tx : txs)
                for (unsigned ty : tys)
                    if (tx < ntx && ty < nty) lists[c][tx + ntx * ty].push_back(e);
        }
        for (const auto& l : lists[c]) most = std::max(most, l.size());
    }
    if (why.empty() && most > 64) why = form == 1 ? "more than 64 sources in one tile" : "more than 64 sources in one column";
    if (!why.empty()) {
        h->bands.clear();
        return autom ? 0 : fail(EMS_E_ARG, "fused step unavailable: " + why);
    }
    int rc;
    for (int c = 0; c < 2; ++c)
        if ((rc = upload_exc_groups(h, deferred[c], h->exc_def[c]))) return rc;
    if (!cells.empty()) {
        if ((rc = upload(h, &h->cell_list, cells.data(), cells.size()))) return rc;
        h->ncells = (unsigned)cells.size();
    }
    for (int side = 0; side < 2; ++side) {
        h->nrim[side] = 0;
        if (h->mur_fold[side] < 0) continue;
        // points z * Ny + y of an x face with y or z within 2 lines of the edge
        std::vector<unsigned> rim;
        for (unsigned z = 0; z < Nz; ++z)
            for (unsigned y = 0; y < Ny; ++y)
                if (y < 2 || y + 2 >= Ny || z < 2 || z + 2 >= Nz) rim.push_back(z * Ny + y);
        if ((rc = upload(h, &h->mur_rim[side], rim.data(), rim.size()))) return rc;
        h->nrim[side] = (unsigned)rim.size();
    }
    for (int c = 0; c < 2; ++c) {
        std::vector<unsigned> beg(nlists + 1, 0);
        std::vector<ExcEnt> ent;
        for (unsigned t = 0; t < nlists; ++t) {
            ent.insert(ent.end(), lists[c][t].begin(), lists[c][t].end());
            beg[t + 1] = (unsigned)ent.size();
            // form 3: the entries of each group of four columns (one quad)
            // ordered by plane, list order kept within a plane
            if (form == 3 && t % 4 == 3)
                std::stable_sort(ent.begin() + beg[t - 3], ent.end(),
                                 [](const ExcEnt& l, const ExcEnt& r) { return l.z < r.z; });
        }
        ExcArgs& E = c ? h->eI : h->eV;
        unsigned* db;
        ExcEnt* de;
        if ((rc = upload(h, &db, beg.data(), beg.size())) || (rc = upload(h, &de, ent.data(), ent.size()))) return rc;
        E.beg = db;
        E.ent = de;
        E.sig = h->sig[c];
        E.length = h->sigLen;
        E.period = h->period;
    }
    // second buffers for state n+1; cells a step does not write (the last
    // current line of each direction) must hold the same values in both
    if ((rc = h->alloc(&h->V_alt, 3 * h->cs)) || (rc = h->alloc(&h->I_alt, 3 * h->cs))) return rc;
    HIPCHK(hipMemcpy(h->V_alt, h->V, 3 * h->cs * sizeof(float), hipMemcpyDeviceToDevice));
    HIPCHK(hipMemcpy(h->I_alt, h->I, 3 * h->cs * sizeof(float), hipMemcpyDeviceToDevice));
    for (int side = 0; side < 2; ++side) {
        PmlArgs& P = side ? h->pmlI : h->pmlV;
        if (!P.n) continue;
        if ((rc = h->alloc(&h->flux_alt[side], 3 * P.npos))) return rc;
        HIPCHK(hipMemcpy(h->flux_alt[side], P.flux_in, 3 * P.npos * sizeof(float), hipMemcpyDeviceToDevice));
    }
    HIPCHK(hipDeviceSynchronize());
    h->V_base = h->V;
    if (form == 1) {
        h->ntx = ntx;
        h->nty = nty;
        h->fzdepth = choose_fused_zdepth(ntx * nty, Nz);
        h->fnzc = (Nz + h->fzdepth - 1) / h->fzdepth;
    } else if (form == 3) {
        // tiles of kBlock quads over the plane (k_step4), or of 64 quads x 4
        // rows (k_step4t, rows of at least 64 quads); 8 planes per chunk (128
        // for the tiles: 10.72, 10.61, 10.51 ms per sweep on the Mur layers
        // at 16, 32, 64, and 10.47 against 10.53 at 128), shallower when the
        // grid would give fewer than 2048 workgroups
        const unsigned NQ = Nx / 4;
        h->q4ntq = (NQ + 63) / 64;
        h->ntx = h->q4tile ? h->q4ntq * ((Ny + kQTileRows - 1) / kQTileRows) : (h->g.plane / 4 + kBlock - 1) / kBlock;
        unsigned d = h->q4tile ? 128 : 8;
        while (d > 2 && (unsigned long long)h->ntx * ((Nz + d - 1) / d) < 2048ull) d /= 2;
        if (const char* zd = std::getenv("EMS_Q4ZDEPTH")) {
            const int v = std::atoi(zd);
            if (v >= 1 && v <= 1024) d = (unsigned)v;
        }
        h->fzdepth = d;
        h->fnzc = (Nz + d - 1) / d;
    } else {
        // the two-half-step tiles (kBlock consecutive columns) and z depth
        h->fzdepth = h->g.zdepth;
        h->fnzc = h->g.nzc;
    }
    h->fused = form;
    return 0;
}

int ems_set_fused(ems_engine* h, int mode)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (mode < -1 || mode > 3)
        return fail(EMS_E_ARG, "step form is -1 (auto), 0 (two half steps), 1 (LDS sweep) or 2 (column sweep)");
    h->fused_req = mode;
    return 0;
}

int ems_get_fused(const ems_engine* h, int* fused, unsigned* zdepth)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (fused) *fused = h->fused;
    if (zdepth) *zdepth = h->fused ? h->fzdepth : h->g.zdepth;
    return 0;
}

int ems_set_steady_state(ems_engine* h, unsigned period_steps, unsigned nprobe, const int* dir, const unsigned* pos,
                         unsigned history_capacity)
{
    if (!h || !dir || !pos) return fail(EMS_E_ARG, "null argument");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (h->has_ss) return fail(EMS_E_STATE, "steady-state detection already set");
    if (period_steps == 0 || nprobe == 0) return fail(EMS_E_ARG, "empty period or probe list");
    std::vector<unsigned long long> lin(nprobe);
    for (unsigned k = 0; k < nprobe; ++k) {
        const unsigned x = pos[k], y = pos[nprobe + k], z = pos[2 * nprobe + k];
        if (dir[k] < 0 || dir[k] > 2 || x >= h->N[0] || y >= h->N[1] || z >= h->N[2])
            return fail(EMS_E_ARG, "steady-state probe outside the mesh");
        lin[k] = (unsigned long long)dir[k] * h->cs + h->lin(x, y, z);
    }
    HIPCHK(hipSetDevice(h->device));
    SteadyDev S{};
    S.n = nprobe;
    S.p = period_steps;
    S.cap = std::max(1u, history_capacity);
    unsigned long long* dl;
    int rc;
    if ((rc = upload(h, &dl, lin.data(), nprobe)) || (rc = h->alloc(&S.rec, (size_t)nprobe * 2 * period_steps)) ||
        (rc = h->alloc(&S.state, 3)) || (rc = h->alloc(&S.hist_ts, S.cap)) || (rc = h->alloc(&S.hist_diff, S.cap)) ||
        (rc = h->alloc(&h->ss_part, 2 * 1024)))
        return rc;
    S.lin = dl;
    HIPCHK(hipMemset(S.rec, 0, (size_t)nprobe * 2 * period_steps * sizeof(float)));
    const double st[3] = {1.0, 0.0, 0.0};
    HIPCHK(hipMemcpy(S.state, st, sizeof(st), hipMemcpyHostToDevice));
    h->ss = S;
    h->h_ss = std::move(lin);
    h->has_ss = true;
    return 0;
}

int ems_steady_state(ems_engine* h, double* last_max_diff, unsigned* evaluations, unsigned* ts, double* diff,
                     unsigned cap)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (!h->has_ss) return fail(EMS_E_STATE, "no steady-state detection");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    double st[3];
    HIPCHK(hipMemcpy(st, h->ss.state, sizeof(st), hipMemcpyDeviceToHost));
    if (last_max_diff) *last_max_diff = st[0];
    const unsigned n = (unsigned)st[2];
    if (evaluations) *evaluations = n;
    const unsigned m = std::min(std::min(n, h->ss.cap), cap);
    if (ts && m) HIPCHK(hipMemcpy(ts, h->ss.hist_ts, m * sizeof(unsigned), hipMemcpyDeviceToHost));
    if (diff && m) HIPCHK(hipMemcpy(diff, h->ss.hist_diff, m * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

// Quad half steps (k_volt4 / k_curr4): two-half-step engines whose rows hold
// a whole number of four-cell groups.  Automatic mode takes them on meshes
// without UPML (1024 x 1024 x 768 Mur layers: 6.37 -> 5.79 ms per half
// step).  On a UPML mesh, quads run as two launches: the box without UPML
// cells without UPML code, the six boxes around it with it.  Automatic mode
// keeps one cell per lane there: on the 256^3 UPML bricks the UPML-free box
// (82 % of the cells) takes 119 us, but the quads' UPML path over the
// remaining 18 % takes 75 us, against 161 us for the whole mesh at one cell
// per lane.  z depth: 4 planes per workgroup, shallower when the grid would
// give fewer than 2048 workgroups.
static int setup_quad(ems_engine* h)
{
    h->quad = false;
    if (h->quad_req == 0) return 0;
    std::string why;
    if (h->fused) why = "the single-sweep step forms have no quad form";
    else if (h->N[0] % 4) why = "the number of x lines is not a multiple of 4";
    if (!why.empty()) return h->quad_req == 1 ? fail(EMS_E_ARG, "quad half steps unavailable: " + why) : 0;
    GridDesc& q = h->gq;
    q = h->g;
    q.tx = 0;
    q.ntx = 0;
    q.qtiles = (q.plane / 4 + kBlock - 1) / kBlock;
    unsigned d = 4;
    while (d > 1 && (unsigned long long)q.qtiles * ((q.Nz + d - 1) / d) < 2048ull) d /= 2;
    if (const char* zd = std::getenv("EMS_QZDEPTH")) {
        const int v = std::atoi(zd);
        if (v >= 1 && v <= 1024) d = (unsigned)v;
    }
    q.zdepth = d;
    q.nzc = (q.Nz + d - 1) / d;
    const unsigned NQ = h->N[0] / 4;
    // boxes in quads x rows x planes; workgroups counted box after box
    QBox hb[3][kMaxQBoxes] = {};          // all, in, out
    unsigned nb[3] = {0, 0, 0}, blk[3] = {0, 0, 0};
    // the boxes around the UPML-free box hold few cells and the longer UPML
    // update: one plane per workgroup, for enough waves to hide its latency
    unsigned dout = 1;
    if (const char* zo = std::getenv("EMS_QZOUT")) {
        const int v = std::atoi(zo);
        if (v >= 1 && v <= 1024) dout = (unsigned)v;
    }
    auto add = [&](int set, unsigned qa, unsigned nq, unsigned ya, unsigned ny, unsigned za, unsigned zb) {
        if (!nq || !ny || za >= zb) return;
        QBox& b = hb[set][nb[set]++];
        b.qa = qa;
        b.nq = nq;
        b.ya = ya;
        b.ny = ny;
        b.za = za;
        b.zb = zb;
        b.zd = set == 2 ? dout : d;
        b.ntiles = (nq * ny + kBlock - 1) / kBlock;
        b.first = blk[set];
        blk[set] += b.ntiles * ((zb - za + b.zd - 1) / b.zd);
    };
    add(0, 0, NQ, 0, h->N[1], 0, h->N[2]);
    // UPML mesh: the largest box of whole quads holding no UPML cell, found
    // along the mesh's centre lines, and the six boxes around it
    h->qsplit = false;
    if (h->pmlV.n) {
        const PmlArgs& P = h->pmlV;
        const unsigned c[3] = {h->N[0] / 2, h->N[1] / 2, h->N[2] / 2};
        unsigned lo[3], hi[3];                  // interior [lo, hi) per axis
        for (int a = 0; a < 3; ++a) {
            auto in_slab = [&](unsigned v) {
                unsigned p[3] = {c[0], c[1], c[2]};
                p[a] = v;
                for (int s = 0; s < P.n; ++s) {
                    const SlabTab& S = P.tab[s];
                    if ((int)p[0] >= S.x0 && (int)p[0] <= S.x1 && (int)p[1] >= S.y0 && (int)p[1] <= S.y1 &&
                        (int)p[2] >= S.z0 && (int)p[2] <= S.z1)
                        return true;
                }
                return false;
            };
            lo[a] = 0;
            while (lo[a] < h->N[a] && in_slab(lo[a])) ++lo[a];
            hi[a] = h->N[a];
            while (hi[a] > lo[a] && in_slab(hi[a] - 1)) --hi[a];
        }
        const unsigned qa = (lo[0] + 3) / 4, qb = hi[0] / 4;
        bool ok = qa < qb && lo[1] < hi[1] && lo[2] < hi[2];
        // no slab may reach into the box
        for (int s = 0; s < P.n && ok; ++s) {
            const SlabTab& S = P.tab[s];
            const bool meet = S.x0 < (int)(4 * qb) && S.x1 >= (int)(4 * qa) && S.y0 < (int)hi[1] &&
                              S.y1 >= (int)lo[1] && S.z0 < (int)hi[2] && S.z1 >= (int)lo[2];
            if (meet) ok = false;
        }
        if (ok) {
            add(1, qa, qb - qa, lo[1], hi[1] - lo[1], lo[2], hi[2]);
            const unsigned Ny = h->N[1], Nz = h->N[2];
            add(2, 0, NQ, 0, Ny, 0, lo[2]);                        // planes below
            add(2, 0, NQ, 0, Ny, hi[2], Nz);                       // planes above
            add(2, 0, NQ, 0, lo[1], lo[2], hi[2]);                 // rows in front
            add(2, 0, NQ, hi[1], Ny - hi[1], lo[2], hi[2]);        // rows behind
            add(2, 0, qa, lo[1], hi[1] - lo[1], lo[2], hi[2]);     // quads left
            add(2, qb, NQ - qb, lo[1], hi[1] - lo[1], lo[2], hi[2]);  // quads right
            h->qsplit = true;
        }
    }
    if (!h->qbox_dev) {
        int rc;
        if ((rc = h->alloc(&h->qbox_dev, 3 * kMaxQBoxes))) return rc;
    }
    HIPCHK(hipMemcpy(h->qbox_dev, hb, sizeof(hb), hipMemcpyHostToDevice));
    h->qbox_all = QBoxes{h->qbox_dev, nb[0]};
    h->qbox_in = QBoxes{h->qbox_dev + kMaxQBoxes, nb[1]};
    h->qbox_out = QBoxes{h->qbox_dev + 2 * kMaxQBoxes, nb[2]};
    h->qblk_all = blk[0];
    h->qblk_in = blk[1];
    h->qblk_out = blk[2];
    if (const char* sp = std::getenv("EMS_QSPLIT")) h->qsplit = h->qsplit && std::atoi(sp) != 0;
    // automatic mode: quads on meshes without UPML
    if (h->quad_req == -1 && h->pmlV.n) return 0;
    h->quad = true;
    return 0;
}

// Voltage sources added by the half-step voltage kernel itself (k_volt4 per
// quad, k_volt per column) when no hook runs between the voltage update and
// the excitation (Mur post and apply, lumped RLC, Lorentz, the steady-state
// record): one launch less per step.  Lists per quad or column, ordered by
// plane, list order kept within a plane.
static int setup_vsrc(ems_engine* h)
{
    h->qsrc = ExcArgs{};
    bool on = !h->fused && h->exc[0].G && h->exc[0].host.size() == h->exc[0].K && h->mur.empty() &&
              h->lor.empty() && h->rlc.empty() && !h->has_ss && h->N[0] < 65535 && h->N[1] < 65535 &&
              h->N[2] < 65535;
    if (const char* qs = std::getenv("EMS_QSRC")) on = on && std::atoi(qs) != 0;
    if (!on) return 0;
    const unsigned w = h->quad ? 4u : 1u;            // cells per list along x
    const unsigned nx = h->N[0] / w;
    const unsigned nl = (unsigned)(h->g.plane / w);
    std::vector<std::vector<ExcEnt>> lists(nl);
    for (const auto& e : h->exc[0].host) lists[e.x / w + nx * (unsigned)e.y].push_back(e);
    std::vector<unsigned> beg(nl + 1, 0);
    std::vector<ExcEnt> ent;
    for (unsigned i = 0; i < nl; ++i) {
        std::stable_sort(lists[i].begin(), lists[i].end(), [](const ExcEnt& l, const ExcEnt& r) { return l.z < r.z; });
        ent.insert(ent.end(), lists[i].begin(), lists[i].end());
        beg[i + 1] = (unsigned)ent.size();
    }
    unsigned* db;
    ExcEnt* de;
    unsigned* dm = nullptr;
    int rc;
    if ((rc = upload(h, &db, beg.data(), beg.size())) || (rc = upload(h, &de, ent.data(), ent.size()))) return rc;
    if (w == 1 && h->g.tx == 0) {
        // k_volt: tiles of kBlock consecutive columns (the single engine's tile
        // shape); only tiles holding a source read the lists
        const unsigned nt = (unsigned)((h->g.plane + kBlock - 1) / kBlock);
        std::vector<unsigned> mask((nt + 31) / 32, 0u);
        for (const auto& e : h->exc[0].host) {
            const unsigned t = (unsigned)(((unsigned long long)e.x + (unsigned long long)h->N[0] * e.y) / kBlock);
            mask[t >> 5] |= 1u << (t & 31);
        }
        if ((rc = upload(h, &dm, mask.data(), mask.size()))) return rc;
    }
    h->qsrc = ExcArgs{db, de, h->sig[0], h->sigLen, h->period, dm};
    return 0;
}

}  // extern "C"

// Tile and chunk of k_pair.  A CU holds `waves` wavefronts of the kernel and
// its LDS.  A plane of a workgroup takes at least its round trip (LDS
// exchange, barrier, the loads that did not arrive) and, with the CU full,
// its share of issue and memory time, which grows as rows get short: every
// row of a tile starts and ends inside a cache line.  Measured per plane and
// 1024 columns: 2.81, 2.09, 1.76 us at 39, 64 and 128 columns a row (253 x
// 209 x 178 cavity, from HBM), and with UPML 2.49, 2.38, 2.05, 1.65 us per
// 512 at 23, 36, 53 and 102.  The estimate adds the planes and columns that
// neighbours compute twice and the last, partly empty round of workgroups;
// the smallest wins.
// tiles of t lines, advancing by t-3, that cover n lines
static unsigned pair_tiles(unsigned n, unsigned t) { return n <= t ? 1u : (n - 3u + t - 4u) / (t - 3u); }

struct PairCost {
    double lat, issue, row;        // us: a plane's round trip; per 1024 columns; and that over the row length
};
constexpr PairCost kPairPlain{0.9, 1.3, 59.0}, kPairUpml{1.5, 2.8, 50.0};
static void choose_pair_tile(const unsigned N[3], const PairCost& cost, unsigned most, unsigned column, unsigned waves,
                             size_t table, unsigned cus, PairArgs& a)
{
    double best = 1e300;
    // lines per tile that cover n lines evenly with k tiles
    auto even = [](unsigned n, unsigned k) { return k == 1 ? n : (n - 3u + k - 1u) / k + 3u; };
    unsigned ltx = 0;
    for (unsigned kx = 1; kx <= N[0]; ++kx) {
        const unsigned tx = even(N[0], kx), nx = pair_tiles(N[0], tx);
        if (tx < std::min(N[0], 24u)) break;
        if (tx == ltx || tx > 256) continue;
        ltx = tx;
        unsigned lty = 0;
        for (unsigned ky = 1; ky <= N[1]; ++ky) {
            const unsigned ty = even(N[1], ky), ny = pair_tiles(N[1], ty);
            if (ty < std::min(N[1], 6u)) break;
            if (ty == lty) continue;
            lty = ty;
            const unsigned T = (tx * ty + 63u) / 64u * 64u;
            const size_t lds = (size_t)column * T + table;
            if (T > most || lds > kLdsBytes) continue;
            const unsigned res = std::min(waves / (T / 64u), (unsigned)(kLdsBytes / lds));
            if (!res) continue;
            unsigned last = 0;
            for (unsigned nz = 1; nz <= N[2]; ++nz) {
                const unsigned zd = (N[2] + nz - 1) / nz;
                if (zd == last) continue;
                last = zd;
                if (zd < 2 && N[2] > 2) break;
                const unsigned long long wg = (unsigned long long)nx * ny * ((N[2] + zd - 1) / zd);
                const unsigned long long rounds = (wg + (unsigned long long)cus * res - 1) / ((unsigned long long)cus * res);
                const double full = (double)std::min<unsigned long long>(res, (wg + cus - 1) / cus) * T / kPairMax;
                const double c = (double)rounds * (zd + 5) * std::max(cost.lat, (cost.issue + cost.row / tx) * full);
                if (c < best) {
                    best = c;
                    a.tx = tx;
                    a.ty = ty;
                    a.ntx = nx;
                    a.ntiles = nx * ny;
                    a.zd = zd;
                }
            }
        }
    }
}

template <int PM>
static const void* pair_kernel(bool cmp, bool lt)
{
    if (!cmp) return (const void*)k_pair<PM, false, false>;
    return lt ? (const void*)k_pair<PM, true, true> : (const void*)k_pair<PM, true, false>;
}

static const void* pair_kernel(const ems_engine* h, bool lt)
{
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    return pm == kPmlCompressed ? pair_kernel<kPmlCompressed>(h->cmp, lt)
           : pm == kPmlPlain    ? pair_kernel<kPmlPlain>(h->cmp, lt)
                                : pair_kernel<kNoPml>(h->cmp, lt);
}

// Two timesteps per launch (k_pair): the automatic step of meshes whose only
// extensions are UPML and sources (Mur, Lorentz, lumped RLC and steady-state
// detection have hooks between the half steps), where neither the step form
// nor the lane width was asked for, 32-bit byte offsets reach every cell and
// the second copy of fields and fluxes fits with 1 GiB to spare.  With UPML
// from a million cells on: per step 31.8 -> 24.4 us at 109 x 97 x 131, 63.5 ->
// 44.5 us at 160 x 150 x 140, 315 -> 218 us at 256^3, but 10.5 -> 12.8 us at
// 64^3, where a workgroup sweeps few planes and most of them are graded; equal
// at 80^3 (16.9 us), 20.6 -> 18.7 us at 90^3.  Flat and long meshes above the
// line: 400 x 400 x 24 78.6 -> 79.5 us, 24 x 400 x 400 93 -> 71, 400 x 24 x 400
// 75 -> 64, 1000 x 1000 x 20 520 -> 402, 50 x 50 x 500 33.9 -> 24.6, 300 x 60 x
// 60 25.5 -> 23.6.  Without UPML at every size: 7.1 -> 5.6 us at 64^3, 34.5 ->
// 14.4 us at 140^3, 103 -> 56 us at 253 x 209 x 178 (plain accesses; 149 to
// 174 us as it ran), also from 4^3 on and for plates and rods.
// Sources in a volume with UPML below four million cells: a pair's updates take
// a column's entries of a plane one after another, the current sources of half
// steps have a launch of their own.  Blocks of 0.3 of the lines along each axis,
// half steps against pairs: three components 51 : 72 us at 110 x 105 x 100, 109
// : 128 at 160 x 150 x 140, 825 : 326 at 256^3; one component 36 : 38, 80 : 68,
// 514 : 244; currents of three components 31 : 67 at 110 x 105 x 100, of one 30
// : 37, 67 : 70 and 320 : 236.  Sheets hold fewer entries and gain (two
// components, 109 x 97 x 131: 106 : 43 normal to x, 103 : 46 to y).  So half
// steps where the voltage entries and twice the current entries exceed a 25th
// of the cells.
constexpr unsigned long long kPairUpmlCells = 1000000, kPairVolumeCells = 4000000;
static int build_pair(ems_engine* h)
{
    h->pair = false;
    const unsigned* N = h->N;
    bool on = (!h->fused || h->fused == 3) && h->fused_req == -1 && h->quad_req == -1 && h->mur.empty() &&
              h->lor.empty() && h->rlc.empty() && !h->has_ss && N[0] < 65535 && N[1] < 65535 && N[2] < 65535 &&
              N[0] >= 4 && N[1] >= 4 && N[2] >= 2 && h->cs < (1ull << 30) && h->pmlV.npos < (1ull << 30);
    const unsigned long long cells = (unsigned long long)h->g.plane * N[2];
    const unsigned long long entries = (unsigned long long)h->exc[0].K + 2ull * h->exc[1].K;
    bool big = !h->pmlV.n || (cells >= kPairUpmlCells && (cells >= kPairVolumeCells || 25ull * entries <= cells));
    for (int c = 0; c < 2; ++c) on = on && h->exc[c].host.size() == h->exc[c].K && h->exc[c].K < kSingle;
    if (const char* e = std::getenv("EMS_PAIR")) big = std::atoi(e) != 0;
    if (!on || !big) return 0;
    const size_t np = h->pmlV.n ? h->pmlV.npos : 0;
    size_t freeb = 0, totalb = 0;
    const size_t need = 6 * ((h->fused ? 0 : h->cs) + np) * sizeof(float) + (1ull << 30);
    if (hipMemGetInfo(&freeb, &totalb) != hipSuccess || freeb < need) return 0;
    PairArgs& a = h->pargs;
    a = PairArgs{};
    a.Nx = N[0];
    a.Ny = N[1];
    a.Nz = N[2];
    a.plane = h->g.plane;
    a.cs = h->cs;
    a.kV = h->kV;
    a.kI = h->kI;
    int rc;
    if (np) {
        SlabTab* tab;
        if ((rc = upload(h, &tab, h->pmlV.tab, (size_t)h->pmlV.n))) return rc;
        a.pml = PairPml{tab, (unsigned)h->pmlV.n, h->pmlV.npos, h->pmlV.pidx, h->pmlV.coef, h->pmlI.coef, h->pmlV.ptab, h->pmlI.ptab};
    }
    // both sides' tables in LDS where they leave it room for the tiles
    size_t table = h->cmp ? (size_t)(h->kV.ntab + h->kI.ntab) * sizeof(float4) : 0;
    const bool lt = h->cmp && table <= kLdsTabBytes;
    if (!lt) table = 0;
    const void* k = pair_kernel(h, lt);
    const unsigned most = np ? kPairMaxPml : kPairMax;
    const unsigned lds = kPairLds * (unsigned)sizeof(float);       // per column
    hipFuncAttributes fa{};
    HIPCHK(hipFuncGetAttributes(&fa, k));
    const unsigned waves = std::min(32u, 4u * (512u / std::max(8u, ((unsigned)fa.numRegs + 7u) / 8u * 8u)));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, h->device));
    choose_pair_tile(N, np ? kPairUpml : kPairPlain, most, lds, waves, table, (unsigned)prop.multiProcessorCount, a);
    if (const char* e = std::getenv("EMS_PAIR_TILE")) {
        unsigned tx, ty, zd;
        if (std::sscanf(e, "%u,%u,%u", &tx, &ty, &zd) == 3 && tx >= 4 && ty >= 4 && tx * ty <= most && zd >= 1) {
            a.tx = std::min(tx, N[0]);
            a.ty = std::min(ty, N[1]);
            a.zd = std::min(zd, N[2]);
            a.ntx = pair_tiles(N[0], a.tx);
            a.ntiles = a.ntx * pair_tiles(N[1], a.ty);
        }
    }
    if (!a.tx) return 0;
    h->pair_threads = (a.tx * a.ty + 63u) / 64u * 64u;
    h->pair_blocks = a.ntiles * ((N[2] + a.zd - 1) / a.zd);
    h->pair_lds = (size_t)lds * h->pair_threads + table;
    // a limit of the kernel, not of this engine: engines of other tiles share it
    HIPCHK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    // sources: lists per column ordered by plane, their planes, and the tiles
    // (rims included) that hold one
    std::vector<unsigned> mask((a.ntiles + 31) / 32, 0u);
    const unsigned nty = a.ntiles / a.ntx;
    // first and last of the n tiles of t lines that hold line x
    auto tiles_of = [](unsigned x, unsigned t, unsigned n) {
        return std::make_pair(x < t ? 0u : (x - t) / (t - 3u) + 1u, std::min(x / (t - 3u), n - 1u));
    };
    bool any = false;
    for (int c = 0; c < 2; ++c) {
        const auto& host = h->exc[c].host;
        PairSrc& S = c ? a.sI : a.sV;
        S = PairSrc{1u, 0u, nullptr, ExcArgs{}};
        if (host.empty()) continue;
        any = true;
        std::vector<unsigned> beg(h->g.plane + 1, 0);
        unsigned lo = ~0u, hi = 0;
        for (const auto& e : host) {
            ++beg[e.x + N[0] * (unsigned)e.y + 1];
            lo = std::min(lo, (unsigned)e.z);
            hi = std::max(hi, (unsigned)e.z);
            const std::pair<unsigned, unsigned> tx = tiles_of(e.x, a.tx, a.ntx), ty = tiles_of(e.y, a.ty, nty);
            for (unsigned j = ty.first; j <= ty.second; ++j)
                for (unsigned i = tx.first; i <= tx.second; ++i) {
                    const unsigned t = i + a.ntx * j;
                    mask[t >> 5] |= 1u << (t & 31);
                }
        }
        for (size_t i = 1; i < beg.size(); ++i) beg[i] += beg[i - 1];
        std::vector<ExcEnt> ent(host.size());
        std::vector<unsigned> at(beg);
        for (const auto& e : host) ent[at[e.x + N[0] * (unsigned)e.y]++] = e;
        auto below = [](const ExcEnt& l, const ExcEnt& r) { return l.z < r.z; };
        std::vector<uint2> cols(h->g.plane);
        for (size_t i = 0; i < h->g.plane; ++i) {
            const auto b = ent.begin() + beg[i], e = ent.begin() + beg[i + 1];
            if (!std::is_sorted(b, e, below)) std::stable_sort(b, e, below);
            const unsigned n = (unsigned)(e - b), first = n ? b->z : 0u;
            bool single = true;
            for (unsigned k = 0; k < n && single; ++k) single = b[k].z == first + k;
            cols[i] = single ? make_uint2(beg[i] | kSingle, first << 16 | n) : make_uint2(beg[i], n);
        }
        uint2* dc;
        ExcEnt* de;
        if ((rc = upload(h, &dc, cols.data(), cols.size())) || (rc = upload(h, &de, ent.data(), ent.size()))) return rc;
        S = PairSrc{lo, hi, dc, ExcArgs{nullptr, de, h->sig[c], h->sigLen, h->period, nullptr}};
    }
    if (any) {
        unsigned* dm;
        if ((rc = upload(h, &dm, mask.data(), mask.size()))) return rc;
        a.tmask = dm;
    }
    // every pair writes all of state n+2 (UPML padding positions stay zero);
    // the quad sweep has its second buffers already
    if (!h->fused) {
        if ((rc = h->alloc(&h->V_alt, 3 * h->cs)) || (rc = h->alloc(&h->I_alt, 3 * h->cs))) return rc;
        HIPCHK(hipMemset(h->V_alt, 0, 3 * h->cs * sizeof(float)));
        HIPCHK(hipMemset(h->I_alt, 0, 3 * h->cs * sizeof(float)));
    }
    for (int side = 0; side < 2 && np; ++side) {
        if ((rc = h->alloc(&h->flux_alt[side], 3 * np))) return rc;
        HIPCHK(hipMemset(h->flux_alt[side], 0, 3 * np * sizeof(float)));
    }
    HIPCHK(hipStreamSynchronize(nullptr));       // the fills; not other engines' streams
    h->numts_alt = h->numts_dev + 2;
    h->V_base = h->V;
    h->pair = true;
    return 0;
}

// what was free may have been taken meanwhile: single steps then
static int setup_pair(ems_engine* h)
{
    const size_t n = h->allocs.size();
    const int rc = build_pair(h);
    if (rc != EMS_E_NOMEM) return rc;
    while (h->allocs.size() > n) h->release(h->allocs.size() - 1);
    if (!h->fused) h->V_alt = h->I_alt = nullptr;
    h->flux_alt[0] = h->flux_alt[1] = nullptr;
    h->pargs = PairArgs{};
    return 0;
}

// ---------------------------------------------------------------------------
// Hook launches (k_hooks): the jobs of a phase in the reference's order, each
// put into the phase's last launch unless it touches a field element that a
// job of that launch sets, or sets one that a job of that launch touches.
// ---------------------------------------------------------------------------
namespace {

struct HookPlan {
    HookJob d{};
    std::vector<unsigned long long> elems;    // sorted component * cs + cell of a list job
    std::vector<unsigned> cells;              // sorted cells that a list job sets all components of
    std::vector<unsigned char> lines[3];      // per axis and line: bit c where component c has such an element
    bool writes = true;                       // it sets field elements
    const ems_engine::MurGeo* mur = nullptr;  // a Mur face's job
    int face = -1;
};

// stable sort by the bits from `lo` on.  Lists of a mesh's cells have millions
// of entries in any order: 4 million keys 27 ms, std::sort 183
void sort_keys(std::vector<unsigned long long>& a, unsigned lo = 0)
{
    constexpr unsigned kBits = 12, kBuckets = 1u << kBits;
    auto less = [lo](unsigned long long l, unsigned long long r) { return l >> lo < r >> lo; };
    if (std::is_sorted(a.begin(), a.end(), less)) return;
    if (a.size() < 4 * kBuckets) {
        std::stable_sort(a.begin(), a.end(), less);
        return;
    }
    const unsigned long long top = *std::max_element(a.begin(), a.end());
    std::vector<unsigned long long> b(a.size());
    for (unsigned s = lo; s < 64 && top >> s; s += kBits) {
        size_t at[kBuckets + 1] = {};
        for (unsigned long long k : a) ++at[(k >> s & (kBuckets - 1)) + 1];
        for (unsigned d = 0; d < kBuckets; ++d) at[d + 1] += at[d];
        for (unsigned long long k : a) b[at[k >> s & (kBuckets - 1)]++] = k;
        a.swap(b);
    }
}

// the lines that a list job's elements lie on
void find_lines(const ems_engine* h, HookPlan& q)
{
    for (int n = 0; n < 3; ++n) q.lines[n].assign(h->N[n], 0);
    auto mark = [&](unsigned p, unsigned char bits) {
        const unsigned z = p / h->g.plane, r = p - z * h->g.plane, y = r / h->N[0];
        q.lines[0][r - y * h->N[0]] |= bits;
        q.lines[1][y] |= bits;
        q.lines[2][z] |= bits;
    };
    for (unsigned long long e : q.elems) {
        const unsigned c = e >= 2 * h->cs ? 2u : e >= h->cs ? 1u : 0u;
        mark((unsigned)(e - c * h->cs), (unsigned char)(1u << c));
    }
    for (unsigned p : q.cells) mark(p, 7);
}

// whether two list jobs share an element
bool share_element(const ems_engine* h, const HookPlan& a, const HookPlan& b)
{
    for (size_t i = 0, j = 0; i < a.elems.size() && j < b.elems.size();) {
        if (a.elems[i] == b.elems[j]) return true;
        if (a.elems[i] < b.elems[j]) ++i;
        else ++j;
    }
    auto in_cells = [h](const std::vector<unsigned long long>& e, const std::vector<unsigned>& c) {
        if (c.size() < e.size() / 3) {
            for (unsigned x : c)
                for (unsigned n = 0; n < 3; ++n)
                    if (std::binary_search(e.begin(), e.end(), n * h->cs + x)) return true;
            return false;
        }
        for (unsigned long long k : e)
            if (std::binary_search(c.begin(), c.end(), (unsigned)(k % h->cs))) return true;
        return false;
    };
    if (in_cells(a.elems, b.cells) || in_cells(b.elems, a.cells)) return true;
    for (size_t i = 0, j = 0; i < a.cells.size() && j < b.cells.size();) {
        if (a.cells[i] == b.cells[j]) return true;
        if (a.cells[i] < b.cells[j]) ++i;
        else ++j;
    }
    return false;
}

// an element of list job l on the line that Mur job m reads (the neighbour
// line, before or after the update; only if l sets it) or sets (the face line)
bool mur_touches(const HookPlan& m, const HookPlan& l)
{
    const auto& on = l.lines[m.mur->ny];
    if (on.empty()) return false;
    const unsigned tangential = 7u & ~(1u << m.mur->ny);
    return (m.d.kind != kMurPost && (on[m.mur->line] & tangential)) ||
           (l.writes && m.d.kind != kMurApply && (on[m.mur->shift] & tangential));
}

bool hooks_conflict(const ems_engine* h, const HookPlan& a, const HookPlan& b)
{
    if (a.d.curr != b.d.curr) return false;
    if (a.mur && b.mur) {
        if (a.face == b.face) return true;               // through the face's own values
        auto hit = [&](const HookPlan& r, const HookPlan& w) {      // w's apply sets what r's post reads
            if (w.d.kind == kMurPost || r.d.kind == kMurApply) return false;
            return r.mur->ny != w.mur->ny || r.mur->shift == w.mur->line;
        };
        if (hit(a, b) || hit(b, a)) return true;
        if (a.d.kind == kMurPost || b.d.kind == kMurPost) return false;
        // two applies setting one element: over[] resolves them
        return (a.mur->ny != b.mur->ny || a.mur->line == b.mur->line) && h->mur.size() > kMurMaskFaces;
    }
    if (a.mur || b.mur) {
        const HookPlan& m = a.mur ? a : b;
        const HookPlan& l = a.mur ? b : a;
        return mur_touches(m, l);
    }
    if (!a.writes && !b.writes) return false;
    return share_element(h, a, b);
}

}  // namespace

// the jobs as launches; `alone` ends a launch after job `alone` (its launch's
// index goes to *at)
static int build_hook_launches(ems_engine* h, const std::vector<HookPlan>& jobs, bool independent,
                               std::vector<HookLaunch>& out, int alone = -1, int* at = nullptr)
{
    out.clear();
    std::vector<std::vector<const HookPlan*>> sets;
    bool closed = true;
    for (size_t j = 0; j < jobs.size(); ++j) {
        if (!jobs[j].d.n) continue;
        bool fresh = closed || sets.back().size() >= kMaxHookJobs;
        for (size_t i = 0; !fresh && !independent && i < sets.back().size(); ++i)
            fresh = hooks_conflict(h, *sets.back()[i], jobs[j]);
        if (fresh) sets.emplace_back();
        sets.back().push_back(&jobs[j]);
        closed = (int)j == alone;
        if (closed && at) *at = (int)sets.size() - 1;
    }
    std::vector<HookJob> d;
    for (const auto& set : sets) {
        HookLaunch L{};
        for (const HookPlan* q : set) {
            L.first[L.n++] = L.nblk;
            L.nblk += (q->d.n + kBlock - 1) / kBlock;
            d.push_back(q->d);
        }
        out.push_back(L);
    }
    if (d.empty()) return 0;
    HookJob* dj;
    int rc = upload(h, &dj, d.data(), d.size());
    for (auto& L : out) {
        L.jobs = dj;
        dj += L.n;
    }
    return rc;
}

// earlier faces (bit: creation index) that set the P (c = 0) or PP component
// of each of face k's points too, appended to `all`; its offset there, or -1
// where there is none
static long mur_over(const ems_engine* h, int k, int c, std::vector<unsigned char>& all)
{
    if (h->mur.size() > kMurMaskFaces) return -1;
    const auto& G = h->mur_geo[k];
    const int nP = (G.ny + 1) % 3, nPP = (G.ny + 2) % 3, comp = c ? nPP : nP;
    const MurDev& m = h->mur[k];
    const bool tr = nP < nPP;             // device order of the points (ems_add_mur)
    const size_t at = all.size();
    for (int j = 0; j < k; ++j) {
        const auto& J = h->mur_geo[j];
        if (J.ny == comp || (J.ny == G.ny && J.line != G.line)) continue;
        all.resize(at + (size_t)m.na * m.nb, 0);
        unsigned a0 = 0, a1 = m.na, b0 = 0, b1 = m.nb;      // where face j meets this one
        if (J.ny == nP) {
            a0 = J.line;
            a1 = J.line + 1;
        } else if (J.ny == nPP) {
            b0 = J.line;
            b1 = J.line + 1;
        }
        for (unsigned a = a0; a < a1; ++a)
            for (unsigned b = b0; b < b1; ++b)
                all[at + (tr ? (size_t)b * m.na + a : (size_t)a * m.nb + b)] |= (unsigned char)(1u << j);
    }
    return all.size() == at ? -1 : (long)at;
}

static int setup_hooks(ems_engine* h)
{
    const int nmur = (int)h->mur.size();
    auto mur_job = [&](int kind, int k) {
        HookPlan q;
        q.d.kind = kind;
        q.d.mur = h->mur[k];
        q.d.n = h->mur[k].na * h->mur[k].nb;
        q.mur = &h->mur_geo[k];
        q.face = k;
        return q;
    };
    auto exc_job = [&](const ems_engine::Exc& e, int curr, int bias) {
        HookPlan q;
        q.d.kind = kExcite;
        q.d.curr = curr;
        q.d.n = e.G;
        q.d.gbeg = e.gbeg;
        q.d.glin = e.glin;
        q.d.amp = e.amp;
        q.d.delay = e.delay;
        q.d.sig = h->sig[curr];
        q.d.length = h->sigLen;
        q.d.period = h->period;
        q.d.ts_bias = bias;
        q.elems = e.h_glin;
        sort_keys(q.elems);
        if (!curr && nmur) find_lines(h, q);
        return q;
    };
    auto folded = [&](int k) { return k == h->mur_fold[0] || k == h->mur_fold[1]; };
    int rc;
    std::vector<unsigned char> over;
    std::vector<long> over_at;
    for (int k = 0; k < nmur; ++k)
        for (int c = 0; c < 2; ++c) over_at.push_back(mur_over(h, k, c, over));
    unsigned char* d_over = nullptr;
    if (!over.empty() && (rc = upload(h, &d_over, over.data(), over.size()))) return rc;
    auto mur_apply = [&](int k) {
        HookPlan q = mur_job(kMurApply, k);
        for (int j = 0; j < nmur && j < (int)kMurMaskFaces; ++j) q.d.start[j] = h->mur[j].start_ts;
        for (int c = 0; c < 2; ++c) q.d.over[c] = over_at[2 * k + c] < 0 ? nullptr : d_over + over_at[2 * k + c];
        return q;
    };
    std::vector<HookPlan> pre, v, c;
    // before the voltage update: nothing here sets a field element.  The
    // current side's ADE reads currents, which nothing sets before the current
    // update, and goes with the hooks after the voltage update
    for (int k = 0; k < nmur; ++k)
        if (!folded(k)) pre.push_back(mur_job(kMurPre, k));
    for (int side = 0; side < 2; ++side)
        for (size_t k = side; k < h->lor.size(); k += 2) {
            if (!(side ? h->lor_i : h->lor_v)[k / 2]) continue;
            HookPlan q;
            q.d.kind = kLorPre;
            q.d.curr = side;
            q.d.n = 3 * h->lor[k].count;
            q.d.lor = h->lor[k];
            (side ? v : pre).push_back(q);
        }
    for (const auto& r : h->rlc) {
        HookPlan q;
        q.d.kind = kRlcPre;
        q.d.n = r.count;
        q.d.rlc = r;
        pre.push_back(q);
    }
    if ((rc = build_hook_launches(h, pre, true, h->hooks_pre))) return rc;
    // beside the current update where that is a launch of plain accesses (with
    // non-temporal ones a step takes 100 us and more, a launch 4); every hook
    // here has one after the voltage update, which leaves it the timestep
    h->pre_ahead = !h->fused && !h->nt_fields && h->hooks_pre.size() == 1;
    if (h->fused && nmur) {
        h->curr_again.clear();
        for (size_t k = 0; k < h->bands.size() || (h->ncells && k == h->bands.size()); ++k) {
            if (h->curr_again.empty() || (k < h->bands.size() && k % kMaxBands == 0)) h->curr_again.push_back(CurrAgain{});
            CurrAgain& A = h->curr_again.back();
            unsigned long long cnt = h->ncells;
            if (k < h->bands.size()) {
                const auto& b = h->bands[k];
                A.band[A.nband++] = CurrBand{b.axis, b.lo, b.hi, A.nblk};
                cnt = (unsigned long long)(b.hi - b.lo + 1) * h->N[0] * h->N[1] * h->N[2] / h->N[b.axis];
                A.first = A.nblk + (unsigned)((cnt + kBlock - 1) / kBlock);
            } else {
                A.cells = h->cell_list;
                A.ncells = h->ncells;
            }
            A.nblk += (unsigned)((cnt + kBlock - 1) / kBlock);
        }
        // beside the currents done again
        h->pre_ahead = !h->curr_again.empty() && h->hooks_pre.size() == 1;
    }
    if (h->fused) {
        // around the quad sweep: posts, applies (the rims of the faces inside
        // the sweep), then the deferred sources; nothing else has a form there
        if (!nmur) return 0;
        for (int k = nmur - 1; k >= 0; --k)
            if (!folded(k)) v.push_back(mur_job(kMurPost, k));
        for (int k = nmur - 1; k >= 0; --k) {
            HookPlan q = mur_apply(k);
            const int side = k == h->mur_fold[0] ? 0 : k == h->mur_fold[1] ? 1 : -1;
            if (side >= 0) {
                q.d.list = h->mur_rim[side];
                q.d.n = h->nrim[side];
            }
            v.push_back(q);
        }
        if (h->exc_def[0].G) v.push_back(exc_job(h->exc_def[0], 0, 0));
        if ((rc = build_hook_launches(h, v, false, h->hooks_v))) return rc;
        if (h->exc_def[1].G) c.push_back(exc_job(h->exc_def[1], 1, 0));
        return build_hook_launches(h, c, false, h->hooks_i);
    }
    // after the voltage update: Mur post (reverse creation order, reads only),
    // steady-state record, lumped RLC, Lorentz, Mur apply (reverse creation
    // order), excitation
    std::vector<HookPlan> list;               // RLC and Lorentz, in order
    for (size_t k = 0; k < h->rlc.size(); ++k) {
        HookPlan q;
        q.d.kind = kRlcApply;
        q.d.n = h->rlc[k].count;
        q.d.rlc = h->rlc[k];
        q.elems = h->h_rlc[k];
        sort_keys(q.elems);
        if (nmur) find_lines(h, q);
        list.push_back(q);
    }
    auto lor_apply = [&](int side, HookPlan& q) {
        // a cell's orders in creation order: keys of the cell and the place in the lists
        std::vector<unsigned long long> keys;
        std::vector<std::pair<size_t, const LorDev*>> from;       // first place of each list
        size_t all = 0;
        for (const auto& l : h->h_lor) all += l.size();
        keys.reserve(all);
        for (size_t k = side; k < h->lor.size(); k += 2) {
            if (!(side ? h->lor_i : h->lor_v)[k / 2]) continue;
            from.push_back({keys.size(), &h->lor[k]});
            for (unsigned x : h->h_lor[k / 2]) keys.push_back((unsigned long long)x << 32 | keys.size());
        }
        if (keys.empty()) return 0;
        if (keys.size() > 0xFFFFFFFFull) return fail(EMS_E_ARG, "too many dispersive cells");
        sort_keys(keys, 32);
        std::vector<unsigned>& cell = q.cells;
        std::vector<unsigned> beg;
        std::vector<LorTerm> term(keys.size());
        for (size_t t = 0; t < keys.size(); ++t) {
            const unsigned x = (unsigned)(keys[t] >> 32), at = (unsigned)keys[t];
            if (cell.empty() || cell.back() != x) {
                cell.push_back(x);
                beg.push_back((unsigned)t);
            }
            size_t f = from.size() - 1;
            while (from[f].first > at) --f;
            term[t] = LorTerm{from[f].second->ade, at - (unsigned)from[f].first, from[f].second->count};
        }
        beg.push_back((unsigned)term.size());
        q.d.kind = kLorApply;
        q.d.curr = side;
        q.d.n = 3 * (unsigned)cell.size();
        if (!side && nmur) find_lines(h, q);
        unsigned *dc, *db;
        LorTerm* dt;
        int r;
        if ((r = upload(h, &dc, cell.data(), cell.size())) || (r = upload(h, &db, beg.data(), beg.size())) ||
            (r = upload(h, &dt, term.data(), term.size())))
            return r;
        q.d.cell = dc;
        q.d.beg = db;
        q.d.term = dt;
        return 0;
    };
    HookPlan lv, li;
    if ((rc = lor_apply(0, lv)) || (rc = lor_apply(1, li))) return rc;
    if (lv.d.n) list.push_back(std::move(lv));
    std::vector<HookPlan> post, apply;
    for (int k = nmur - 1; k >= 0; --k) {
        post.push_back(mur_job(kMurPost, k));
        apply.push_back(mur_apply(k));
    }
    // post and apply as one job where that changes no value read
    bool joint = nmur > 0;
    for (int a = 0; a < nmur && joint; ++a) {
        for (int b = 0; b < nmur && joint; ++b)
            joint = h->mur_geo[a].ny == h->mur_geo[b].ny && h->mur_geo[a].shift != h->mur_geo[b].line &&
                    (a == b || h->mur_geo[a].line != h->mur_geo[b].line);
        for (const auto& q : list) joint = joint && !hooks_conflict(h, post[a], q);
    }
    if (joint)
        for (auto& q : apply) q.d.kind = kMurPostApply;
    else
        v.insert(v.end(), post.begin(), post.end());
    int ss = -1;
    if (h->has_ss) {
        HookPlan q;
        q.d.kind = kSteadyRecord;
        q.d.n = h->ss.n;
        q.d.ss = h->ss;
        q.writes = false;
        q.elems = h->h_ss;
        sort_keys(q.elems);
        if (nmur) find_lines(h, q);
        ss = (int)v.size();
        v.push_back(q);
    }
    v.insert(v.end(), std::make_move_iterator(list.begin()), std::make_move_iterator(list.end()));
    v.insert(v.end(), apply.begin(), apply.end());
    if (h->exc[0].G && !h->qsrc.beg) v.push_back(exc_job(h->exc[0], 0, 0));
    // the steady-state evaluation's energy reads the voltages before any hook sets them
    if ((rc = build_hook_launches(h, v, false, h->hooks_v, ss, &h->hooks_ss))) return rc;
    if (li.d.n) c.push_back(std::move(li));
    if (h->exc[1].G) c.push_back(exc_job(h->exc[1], 1, -1));
    return build_hook_launches(h, c, false, h->hooks_i);
}

extern "C" {

int ems_set_quad(ems_engine* h, int mode)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (h->inited) return fail(EMS_E_STATE, "engine already initialised");
    if (mode < -1 || mode > 1) return fail(EMS_E_ARG, "quad mode is -1 (auto), 0 (off) or 1 (on)");
    h->quad_req = mode;
    return 0;
}

int ems_get_quad(const ems_engine* h, int* on, unsigned* zdepth)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (on) *on = h->quad ? 1 : 0;
    if (zdepth) *zdepth = h->quad ? h->gq.zdepth : 0;
    return 0;
}

int ems_get_pair(const ems_engine* h, int* on, unsigned tile[3], unsigned* launches)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (on) *on = h->pair ? 1 : 0;
    if (tile) {
        tile[0] = h->pair ? h->pargs.tx : 0;
        tile[1] = h->pair ? h->pargs.ty : 0;
        tile[2] = h->pair ? h->pargs.zd : 0;
    }
    if (launches) *launches = h->pair_launches;
    return 0;
}

int ems_init(ems_engine* h)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (h->inited) return 0;
    HIPCHK(hipSetDevice(h->device));
    int rc = upload_upml(h);
    if (rc) return rc;
    if ((rc = setup_fused(h))) return rc;
    if ((rc = setup_quad(h))) return rc;
    if ((rc = setup_vsrc(h))) return rc;
    if ((rc = setup_pair(h))) return rc;
    if ((rc = setup_hooks(h))) return rc;
    h->h_lor = {};               // of the set-up only, four bytes a dispersive cell
    // ems_energy's partial sums: allocated later, they would drop the captured chunks
    if (!h->energy_part && (rc = h->alloc(&h->energy_part, 2 * kEnergyBlocks))) return rc;
    // small compressed tables (both half steps' within 32 KiB) go to LDS in the quad kernels
    h->lds_tab = h->cmp && (size_t)4 * h->n_unique * sizeof(float4) <= kLdsTabBytes;
    if (const char* lt = std::getenv("EMS_LDS_TAB")) h->lds_tab = h->lds_tab && std::atoi(lt) != 0;
    h->inited = true;
    return 0;
}

static void drop_graphs(ems_engine* h);

int ems_add_probe(ems_engine* h, const ems_probe_desc* d, int* id)
{
    if (!h || !d) return fail(EMS_E_ARG, "null argument");
    if (d->type < 0 || d->type > 3) return fail(EMS_E_ARG, "unknown probe type");
    if (d->nelem == 0 || !d->comp || !d->pos) return fail(EMS_E_ARG, "probe without terms");
    if ((d->type == EMS_PROBE_EFIELD || d->type == EMS_PROBE_HFIELD) && (d->nelem != 3 || !d->divisor))
        return fail(EMS_E_ARG, "field probes take three terms with divisors");
    if ((d->type == EMS_PROBE_VOLTAGE || d->type == EMS_PROBE_CURRENT) && !d->sign)
        return fail(EMS_E_ARG, "integral probes need term signs");
    ProbeDev p{};
    p.type = d->type;
    p.nelem = d->nelem;
    p.off = (unsigned)h->h_elin.size();
    p.interval = d->interval;
    p.fd_interval = d->fd_interval;
    p.start_ts = d->start_ts;
    p.stop_ts = d->stop_ts;
    p.capacity = d->capacity;
    for (unsigned e = 0; e < d->nelem; ++e) {
        const unsigned x = d->pos[e], y = d->pos[d->nelem + e], z = d->pos[2 * d->nelem + e];
        if (x >= h->N[0] || y >= h->N[1] || z >= h->N[2] || d->comp[e] > 2)
            return fail(EMS_E_ARG, "probe term outside the mesh");
        h->h_elin.push_back(d->comp[e] * h->cs + h->lin(x, y, z));
        h->h_esign.push_back(d->sign ? (signed char)(d->sign[e] >= 0 ? 1 : -1) : 1);
        h->h_ediv.push_back(d->divisor ? d->divisor[e] : 0.0);
    }
    HIPCHK(hipSetDevice(h->device));
    int rc;
    if ((rc = h->alloc(&p.count, 1)) || (rc = h->alloc(&p.ts_out, std::max(1u, p.capacity))) ||
        (rc = h->alloc(&p.val_out, 3 * (size_t)std::max(1u, p.capacity))))
        return rc;
    HIPCHK(hipMemset(p.count, 0, sizeof(unsigned)));
    h->probes.push_back(p);
    h->probes_dirty = true;
    if (id) *id = (int)h->probes.size() - 1;
    return 0;
}

int ems_probe_results(ems_engine* h, int id, unsigned* count, unsigned* ts, double* values)
{
    if (!h || id < 0 || id >= (int)h->probes.size() || !count) return fail(EMS_E_ARG, "bad probe id");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    const ProbeDev& p = h->probes[id];
    unsigned c = 0;
    HIPCHK(hipMemcpy(&c, p.count, sizeof(unsigned), hipMemcpyDeviceToHost));
    *count = c;
    if (ts && c) HIPCHK(hipMemcpy(ts, p.ts_out, c * sizeof(unsigned), hipMemcpyDeviceToHost));
    if (values && c) HIPCHK(hipMemcpy(values, p.val_out, 3 * (size_t)c * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

}  // extern "C"

// box, field, interpolation and edge lengths of a new dump
static int dump_common(ems_engine* h, int field, int interp, const unsigned start[3], const unsigned stop[3],
                       const double* const edge_len[3], DumpDev& d)
{
    if (!h || !start || !stop || !edge_len) return fail(EMS_E_ARG, "null argument");
    if (field != 0 && field != 1) return fail(EMS_E_ARG, "dump field must be 0 (E) or 1 (H)");
    if (interp < 0 || interp > 2) return fail(EMS_E_ARG, "dump interpolation must be 0 (none), 1 (node) or 2 (cell)");
    for (int n = 0; n < 3; ++n) {
        if (start[n] > stop[n] || stop[n] >= h->N[n]) return fail(EMS_E_ARG, "dump box outside the mesh");
        d.s[n] = start[n];
        d.n[n] = stop[n] - start[n] + 1;
        d.N[n] = h->N[n];
    }
    d.field = field;
    d.interp = interp;
    HIPCHK(hipSetDevice(h->device));
    for (int n = 0; n < 3; ++n) {
        double* de;
        int rc;
        if ((rc = upload(h, &de, edge_len[n], h->N[n]))) return rc;
        d.el[n] = de;
    }
    return 0;
}

extern "C" {

int ems_add_fd_dump(ems_engine* h, int field, int interp, const unsigned start[3], const unsigned stop[3],
                    unsigned fd_interval, unsigned first_ts, unsigned nfreq, unsigned nsamples, const float* factors,
                    const double* const edge_len[3], int* id)
{
    if (!h || !factors) return fail(EMS_E_ARG, "null argument");
    if (fd_interval == 0 || nfreq == 0 || nsamples == 0) return fail(EMS_E_ARG, "empty frequency-domain dump");
    if (first_ts % fd_interval) return fail(EMS_E_ARG, "first dump sample not on the sampling interval");
    DumpDev d{};
    int rc;
    if ((rc = dump_common(h, field, interp, start, stop, edge_len, d))) return rc;
    drop_graphs(h);     // the dump changes the launch pattern of every chunk
    d.fd_interval = fd_interval;
    d.first = first_ts;
    d.nfreq = nfreq;
    d.nsamples = nsamples;
    float* df;
    if ((rc = upload(h, &df, factors, (size_t)nsamples * nfreq * 2))) return rc;
    d.factors = df;
    const size_t npts = (size_t)d.n[0] * d.n[1] * d.n[2];
    if ((rc = h->alloc(&d.acc, (size_t)nfreq * 3 * npts * 2))) return rc;
    HIPCHK(hipMemset(d.acc, 0, (size_t)nfreq * 3 * npts * 2 * sizeof(float)));
    h->dumps.push_back(d);
    h->dump_npts.push_back((unsigned)npts);
    if (id) *id = (int)h->dumps.size() - 1;
    return 0;
}

int ems_fd_dump_results(ems_engine* h, int id, float* out)
{
    if (!h || id < 0 || id >= (int)h->dumps.size() || !out) return fail(EMS_E_ARG, "bad dump id");
    const DumpDev& d = h->dumps[id];
    if (d.td) return fail(EMS_E_ARG, "dump id is a time-domain dump");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipMemcpy(out, d.acc, (size_t)d.nfreq * 3 * h->dump_npts[id] * 2 * sizeof(float), hipMemcpyDeviceToHost));
    return 0;
}

int ems_add_td_dump(ems_engine* h, int field, int interp, const unsigned start[3], const unsigned stop[3],
                    unsigned interval, unsigned start_ts, unsigned stop_ts, unsigned capacity,
                    const double* const edge_len[3], int* id)
{
    if (!h) return fail(EMS_E_ARG, "null argument");
    if (interval == 0 || capacity == 0) return fail(EMS_E_ARG, "empty time-domain dump");
    if (stop_ts < start_ts) return fail(EMS_E_ARG, "dump window ends before it starts");
    DumpDev d{};
    int rc;
    if ((rc = dump_common(h, field, interp, start, stop, edge_len, d))) return rc;
    const unsigned long long first = ((unsigned long long)start_ts + interval - 1) / interval * interval;
    if (first > stop_ts) return fail(EMS_E_ARG, "no sampling step inside the dump window");
    const unsigned long long inwin = ((unsigned long long)stop_ts - first) / interval + 1;
    drop_graphs(h);
    d.td = 1;
    d.fd_interval = interval;
    d.first = (unsigned)first;
    d.nsamples = (unsigned)std::min<unsigned long long>(capacity, inwin);
    const size_t npts = (size_t)d.n[0] * d.n[1] * d.n[2];
    if ((rc = h->alloc(&d.acc, (size_t)d.nsamples * 3 * npts))) return rc;
    HIPCHK(hipMemset(d.acc, 0, (size_t)d.nsamples * 3 * npts * sizeof(float)));
    h->dumps.push_back(d);
    h->dump_npts.push_back((unsigned)npts);
    if (id) *id = (int)h->dumps.size() - 1;
    return 0;
}

int ems_td_dump_results(ems_engine* h, int id, unsigned* count, unsigned* ts, float* out)
{
    if (!h || id < 0 || id >= (int)h->dumps.size() || !count) return fail(EMS_E_ARG, "bad dump id");
    const DumpDev& d = h->dumps[id];
    if (!d.td) return fail(EMS_E_ARG, "dump id is a frequency-domain dump");
    unsigned c = 0;
    if (h->numTS >= d.first && (h->numTS > 0 || h->sampled0))
        c = (unsigned)std::min<unsigned long long>(d.nsamples, (h->numTS - d.first) / d.fd_interval + 1);
    *count = c;
    if (ts)
        for (unsigned k = 0; k < c; ++k) ts[k] = d.first + k * d.fd_interval;
    if (out && c) {
        HIPCHK(hipSetDevice(h->device));
        HIPCHK(hipStreamSynchronize(h->stream));
        HIPCHK(hipMemcpy(out, d.acc, (size_t)c * 3 * h->dump_npts[id] * sizeof(float), hipMemcpyDeviceToHost));
    }
    return 0;
}

static int sync_probe_tables(ems_engine* h)
{
    if (!h->probes_dirty) return 0;
    // captured chunks hold the old probe tables
    drop_graphs(h);
    int rc;
    if ((rc = upload(h, &h->d_probes, h->probes.data(), h->probes.size())) ||
        (rc = upload(h, &h->d_elin, h->h_elin.data(), h->h_elin.size())) ||
        (rc = upload(h, &h->d_esign, h->h_esign.data(), h->h_esign.size())) ||
        (rc = upload(h, &h->d_ediv, h->h_ediv.data(), h->h_ediv.size())))
        return rc;
    h->probes_dirty = false;
    return 0;
}

static bool probe_due(const ems_engine* h, unsigned ts)
{
    for (const auto& p : h->probes) {
        if (ts < p.start_ts || ts > p.stop_ts) continue;
        if ((p.interval && ts % p.interval == 0) || (p.fd_interval && ts % p.fd_interval == 0)) return true;
    }
    return false;
}

static int launch_samples(ems_engine* h)
{
    // ProcessingArray::Process after the step: probes and dumps due at numTS
    if (!h->probes.empty() && probe_due(h, h->numTS)) {
        hipLaunchKernelGGL(k_probe, dim3((unsigned)h->probes.size()), dim3(kBlock), 0, h->stream, h->V, h->I,
                           h->d_probes, h->d_elin, h->d_esign, h->d_ediv, h->numts_dev);
        HIPCHK(hipGetLastError());
    }
    for (size_t k = 0; k < h->dumps.size(); ++k) {
        const DumpDev& d = h->dumps[k];
        unsigned ks;
        if (!dump_sample(d, h->numTS, &ks)) continue;
        const unsigned npts = h->dump_npts[k];
        hipLaunchKernelGGL(k_fd_dump, dim3((npts + kBlock - 1) / kBlock), dim3(kBlock), 0, h->stream,
                           d.field ? h->I : h->V, h->cs, h->N[0], h->g.plane, d, h->numts_dev);
        HIPCHK(hipGetLastError());
    }
    return 0;
}

}  // extern "C"

namespace {

template <int PM, bool CC>
void launch_volt_t(ems_engine* h, unsigned nblk)
{
    if (h->nt_fields)
        hipLaunchKernelGGL((k_volt<PM, CC, true>), dim3(nblk), dim3(kBlock), 0, h->stream, h->g, h->V, h->I, h->kV, h->pmlV,
                           h->qsrc, h->numts_dev);
    else
        hipLaunchKernelGGL((k_volt<PM, CC, false>), dim3(nblk), dim3(kBlock), 0, h->stream, h->g, h->V, h->I, h->kV,
                           h->pmlV, h->qsrc, h->numts_dev);
}

template <int PM, bool CC>
void launch_curr_t(ems_engine* h, unsigned nblk, bool pre)
{
    if (pre)
        hipLaunchKernelGGL((k_curr_pre<PM, CC>), dim3(nblk + h->hooks_pre[0].nblk), dim3(kBlock), 0, h->stream, h->g,
                           h->I, h->V, h->kI, h->pmlI, h->numts_dev, nblk, h->hooks_pre[0]);
    else if (h->nt_fields)
        hipLaunchKernelGGL((k_curr<PM, CC, true>), dim3(nblk), dim3(kBlock), 0, h->stream, h->g, h->I, h->V, h->kI,
                           h->pmlI, h->numts_dev);
    else
        hipLaunchKernelGGL((k_curr<PM, CC, false>), dim3(nblk), dim3(kBlock), 0, h->stream, h->g, h->I, h->V, h->kI,
                           h->pmlI, h->numts_dev);
}

template <bool CC>
void launch_update(ems_engine* h, bool curr, unsigned nblk, bool pre)
{
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    if (pm == kPmlCompressed)
        curr ? launch_curr_t<kPmlCompressed, CC>(h, nblk, pre) : launch_volt_t<kPmlCompressed, CC>(h, nblk);
    else if (pm == kPmlPlain) curr ? launch_curr_t<kPmlPlain, CC>(h, nblk, pre) : launch_volt_t<kPmlPlain, CC>(h, nblk);
    else curr ? launch_curr_t<kNoPml, CC>(h, nblk, pre) : launch_volt_t<kNoPml, CC>(h, nblk);
}

template <int PM, bool CC, bool LT>
void launch_quad_box(ems_engine* h, bool curr, const QBoxes& B, unsigned nblk, unsigned* numts, bool pre)
{
    if (!nblk) return;
    const size_t lds = LT ? (size_t)h->kV.ntab * sizeof(float4) : 0;
    if (curr) {
        if (pre)
            hipLaunchKernelGGL((k_curr4_pre<PM, CC, LT>), dim3(nblk + h->hooks_pre[0].nblk), dim3(kBlock), lds, h->stream,
                               h->gq, B, h->I, h->V, h->kI, h->pmlI, numts, nblk, h->hooks_pre[0]);
        else if (h->nt_fields)
            hipLaunchKernelGGL((k_curr4<PM, CC, true, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, h->gq, B, h->I,
                               h->V, h->kI, h->pmlI, numts);
        else
            hipLaunchKernelGGL((k_curr4<PM, CC, false, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, h->gq, B, h->I,
                               h->V, h->kI, h->pmlI, numts);
    } else {
        if (h->nt_fields)
            hipLaunchKernelGGL((k_volt4<PM, CC, true, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, h->gq, B, h->V,
                               h->I, h->kV, h->pmlV, h->qsrc, h->numts_dev);
        else
            hipLaunchKernelGGL((k_volt4<PM, CC, false, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, h->gq, B, h->V,
                               h->I, h->kV, h->pmlV, h->qsrc, h->numts_dev);
    }
}

template <int PM, bool CC, bool LT>
void launch_quad_lt(ems_engine* h, bool curr, bool pre)
{
    if (PM != kNoPml && h->qsplit) {
        // the box without UPML cells runs without UPML code; the boxes around
        // it (with the timestep counter and the hooks) take the UPML path
        launch_quad_box<kNoPml, CC, LT>(h, curr, h->qbox_in, h->qblk_in, nullptr, false);
        launch_quad_box<PM, CC, LT>(h, curr, h->qbox_out, h->qblk_out, h->numts_dev, pre);
        return;
    }
    launch_quad_box<PM, CC, LT>(h, curr, h->qbox_all, h->qblk_all, h->numts_dev, pre);
}

template <int PM, bool CC>
void launch_quad_t(ems_engine* h, bool curr, bool pre)
{
    if (CC && h->lds_tab) launch_quad_lt<PM, CC, true>(h, curr, pre);
    else launch_quad_lt<PM, CC, false>(h, curr, pre);
}

template <bool CC>
void launch_quad(ems_engine* h, bool curr, bool pre)
{
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    if (pm == kPmlCompressed) launch_quad_t<kPmlCompressed, CC>(h, curr, pre);
    else if (pm == kPmlPlain) launch_quad_t<kPmlPlain, CC>(h, curr, pre);
    else launch_quad_t<kNoPml, CC>(h, curr, pre);
}

// pre: the current update takes the next step's pre hooks along
void dispatch_update(ems_engine* h, bool curr, unsigned nblk, bool pre)
{
    if (h->quad) {
        if (h->cmp) launch_quad<true>(h, curr, pre);
        else launch_quad<false>(h, curr, pre);
        return;
    }
    if (h->cmp) launch_update<true>(h, curr, nblk, pre);
    else launch_update<false>(h, curr, nblk, pre);
}

template <int PM, bool CC>
void launch_step_t(ems_engine* h, const StepArgs& a, unsigned nblk)
{
    hipLaunchKernelGGL((k_step<PM, CC>), dim3(nblk), dim3(kBlock), 0, h->stream, a);
}

void lds_step(ems_engine* h);

}  // namespace

// state n+1 written by a single-sweep step becomes the current state
static void swap_step_buffers(ems_engine* h)
{
    std::swap(h->V, h->V_alt);
    std::swap(h->I, h->I_alt);
    for (int side = 0; side < 2; ++side) {
        PmlArgs& P = side ? h->pmlI : h->pmlV;
        if (!P.n) continue;
        float* cur = const_cast<float*>(P.flux_in);
        P.flux_in = h->flux_alt[side];
        P.flux_out = h->flux_alt[side];
        h->flux_alt[side] = cur;
    }
}

namespace {

template <int PM, bool CC>
void launch_step2_t(ems_engine* h, const Step2Args& a, unsigned nblk)
{
    hipLaunchKernelGGL((k_step2<PM, CC>), dim3(nblk), dim3(kBlock), 0, h->stream, a, h->V, h->I, h->V_alt, h->I_alt,
                       h->pmlV.flux_in, h->flux_alt[0], h->pmlI.flux_in, h->flux_alt[1]);
}

void column_step(ems_engine* h)
{
    Step2Args a{};
    a.g = h->g;
    a.kV = h->kV;
    a.kI = h->kI;
    a.pV = h->pmlV;
    a.pI = h->pmlI;
    a.eV = h->eV;
    a.eI = h->eI;
    a.numts = h->numts_dev;
    const unsigned nblk = h->g.qtiles * h->g.nzc;
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    if (h->cmp) {
        if (pm == kPmlCompressed) launch_step2_t<kPmlCompressed, true>(h, a, nblk);
        else if (pm == kPmlPlain) launch_step2_t<kPmlPlain, true>(h, a, nblk);
        else launch_step2_t<kNoPml, true>(h, a, nblk);
    } else {
        if (pm == kPmlCompressed) launch_step2_t<kPmlCompressed, false>(h, a, nblk);
        else if (pm == kPmlPlain) launch_step2_t<kPmlPlain, false>(h, a, nblk);
        else launch_step2_t<kNoPml, false>(h, a, nblk);
    }
}

template <bool CC, bool LT>
void launch_step4_lt(ems_engine* h, const Step4Args& a, unsigned nblk)
{
    const size_t lds = LT ? (size_t)(h->kV.ntab + h->kI.ntab) * sizeof(float4) : 0;
    if (h->q4tile) {
        if (h->nt_fields)
            hipLaunchKernelGGL((k_step4t<CC, true, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, a, h->V, h->I,
                               h->V_alt, h->I_alt);
        else
            hipLaunchKernelGGL((k_step4t<CC, false, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, a, h->V, h->I,
                               h->V_alt, h->I_alt);
        return;
    }
    if (h->nt_fields)
        hipLaunchKernelGGL((k_step4<CC, true, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, a, h->V, h->I, h->V_alt,
                           h->I_alt);
    else
        hipLaunchKernelGGL((k_step4<CC, false, LT>), dim3(nblk), dim3(kBlock), lds, h->stream, a, h->V, h->I, h->V_alt,
                           h->I_alt);
}

template <bool CC>
void launch_step4_t(ems_engine* h, const Step4Args& a, unsigned nblk)
{
    if (CC && h->lds_tab) launch_step4_lt<CC, true>(h, a, nblk);
    else launch_step4_lt<CC, false>(h, a, nblk);
}

// the quad column sweep over the whole mesh (no UPML)
void quad_step(ems_engine* h)
{
    Step4Args a{};
    a.g = h->g;
    a.kV = h->kV;
    a.kI = h->kI;
    a.eV = h->eV;
    a.eI = h->eI;
    a.numts = h->numts_dev;
    a.qa = 0;
    a.nq = h->N[0] / 4;
    a.ya = 0;
    a.ny = h->N[1];
    a.za = 0;
    a.zb = h->N[2];
    a.xb = h->N[0];
    a.yb = h->N[1];
    a.zdepth = h->fzdepth;
    a.ntiles = h->ntx;
    a.ntq = h->q4ntq;
    for (int side = 0; side < 2; ++side) {
        if (h->mur_fold[side] < 0) continue;
        const MurDev& m = h->mur[h->mur_fold[side]];
        a.mf[side] = MurFold{m.cP, m.cPP, m.mP, m.mPP, m.start_ts, 1u};
    }
    const unsigned nblk = h->ntx * h->fnzc;
    if (h->cmp) launch_step4_t<true>(h, a, nblk);
    else launch_step4_t<false>(h, a, nblk);
}

void launch_hook(ems_engine* h, const HookLaunch& L, float* V, float* I)
{
    hipLaunchKernelGGL(k_hooks, dim3(L.nblk), dim3(kBlock), 0, h->stream, V, I, h->cs, L, h->numts_dev);
}

void launch_hooks(ems_engine* h, const std::vector<HookLaunch>& hooks, float* V, float* I)
{
    for (const auto& L : hooks) launch_hook(h, L, V, I);
}

// one fused step from state n (h->V, h->I, current fluxes) into the second
// buffers, which then become the current state
void fused_step(ems_engine* h, hipEvent_t* ev, bool more, bool& ahead)
{
    // Mur pre hooks read state n (FDTD/engine.cpp:224-265 order; only the quad sweep has Mur)
    if (!ahead) launch_hooks(h, h->hooks_pre, h->V, h->I);
    ahead = more && h->pre_ahead && !ev;
    bool tick = true;
    if (ev) (void)hipEventRecord(ev[0], h->stream);
    if (h->fused == 3) quad_step(h);
    else if (h->fused == 2) column_step(h);
    else lds_step(h);
    if (ev) {
        (void)hipEventRecord(ev[1], h->stream);
        (void)hipEventRecord(ev[2], h->stream);
    }
    if (!h->mur.empty()) {
        // state n+1: Mur post (reverse creation order) on the swept voltages,
        // Mur apply, the deferred voltage sources, then the current update of
        // the planes next to each face again, with their current sources
        launch_hooks(h, h->hooks_v, h->V_alt, h->I_alt);
        for (size_t k = 0; k < h->curr_again.size(); ++k) {
            const CurrAgain& A = h->curr_again[k];
            const bool last = k + 1 == h->curr_again.size();
            const HookLaunch L = last && ahead ? h->hooks_pre[0] : HookLaunch{};
            if (last) tick = !h->hooks_i.empty();
            hipLaunchKernelGGL(k_curr_again, dim3(A.nblk + L.nblk), dim3(kBlock), 0, h->stream, h->g, h->V_alt, h->I,
                               h->I_alt, h->kI, A, L, h->numts_dev, last && !tick ? 1 : 0);
        }
        launch_hooks(h, h->hooks_i, h->V_alt, h->I_alt);
    }
    if (tick) hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, h->stream, h->numts_dev);
    if (ev) (void)hipEventRecord(ev[3], h->stream);
    swap_step_buffers(h);
}

void lds_step(ems_engine* h)
{
    StepArgs a{};
    a.g = h->g;
    a.g.zdepth = h->fzdepth;
    a.g.nzc = h->fnzc;
    a.ntx = h->ntx;
    a.nty = h->nty;
    a.V0 = h->V;
    a.I0 = h->I;
    a.V1 = h->V_alt;
    a.I1 = h->I_alt;
    a.kV = h->kV;
    a.kI = h->kI;
    a.pV = h->pmlV;
    a.pI = h->pmlI;
    if (a.pV.n) a.pV.flux_out = h->flux_alt[0];
    if (a.pI.n) a.pI.flux_out = h->flux_alt[1];
    a.eV = h->eV;
    a.eI = h->eI;
    a.numts = h->numts_dev;
    const unsigned nblk = h->ntx * h->nty * h->fnzc;
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    if (h->cmp) {
        if (pm == kPmlCompressed) launch_step_t<kPmlCompressed, true>(h, a, nblk);
        else if (pm == kPmlPlain) launch_step_t<kPmlPlain, true>(h, a, nblk);
        else launch_step_t<kNoPml, true>(h, a, nblk);
    } else {
        if (pm == kPmlCompressed) launch_step_t<kPmlCompressed, false>(h, a, nblk);
        else if (pm == kPmlPlain) launch_step_t<kPmlPlain, false>(h, a, nblk);
        else launch_step_t<kNoPml, false>(h, a, nblk);
    }
}

}  // namespace

extern "C" {

// one timestep in the reference's hook order (Engine::IterateTS, FDTD/engine.cpp:267-286,
// priorities: UPML > default (lumped RLC, Lorentz, Mur) > excitation); more:
// another one follows before anything else may set a field; ahead: in, the
// step before took this step's pre hooks along; out, this one took the next's
static int launch_step(ems_engine* h, hipEvent_t* ev, bool more, bool& ahead)
{
    if (h->fused) {
        fused_step(h, ev, more, ahead);
        HIPCHK(hipGetLastError());
        return 0;
    }
    const GridDesc& g = h->g;
    const unsigned nblk = g.qtiles * g.nzc;
    // -- pre hooks: Mur, lumped RLC, Lorentz; UPML pre is fused
    if (!ahead) launch_hooks(h, h->hooks_pre, h->V, h->I);
    ahead = more && h->pre_ahead && !ev;
    if (ev) (void)hipEventRecord(ev[0], h->stream);
    dispatch_update(h, false, nblk, false);
    if (ev) (void)hipEventRecord(ev[1], h->stream);
    // -- post and apply hooks: Lorentz pre of the currents, Mur post, steady-state
    //    record (priority +2e6), lumped RLC, Lorentz, Mur apply, excitation
    for (size_t k = 0; k < h->hooks_v.size(); ++k) {
        launch_hook(h, h->hooks_v[k], h->V, h->I);
        if ((int)k == h->hooks_ss && h->numTS % h->ss.p == 0 && h->numTS >= 2 * h->ss.p) {
            const unsigned nb = 1024;
            hipLaunchKernelGGL(k_energy, dim3(nb), dim3(kBlock), 0, h->stream, h->V, h->I, h->cs, h->N[0], h->N[1],
                               h->N[2], h->ss_part);
            hipLaunchKernelGGL(k_ss_eval, dim3(1), dim3(kSsThreads), 0, h->stream, h->ss, h->ss_part, nb, h->numts_dev);
        }
    }
    // -- current half step: fused UPML + update, Lorentz apply, excitation
    if (ev) (void)hipEventRecord(ev[2], h->stream);
    dispatch_update(h, true, nblk, ahead);
    if (ev) (void)hipEventRecord(ev[3], h->stream);
    launch_hooks(h, h->hooks_i, h->V, h->I);
    HIPCHK(hipGetLastError());
    return 0;
}

// state n+2 written by k_pair becomes the current state
static void swap_pair_buffers(ems_engine* h)
{
    swap_step_buffers(h);
    std::swap(h->numts_dev, h->numts_alt);
}

// The engine advances by single steps from now on, on the buffers that hold
// its state now; the ones that only pairs need are freed.
static void leave_pairs(ems_engine* h)
{
    if (!h->pair) return;
    (void)hipStreamSynchronize(h->stream);
    drop_graphs(h);
    h->pair = false;
    auto release = [&](float*& p) {
        for (size_t k = 0; p && k < h->allocs.size(); ++k)
            if (h->allocs[k].p == p) {
                h->release(k);
                p = nullptr;
            }
    };
    if (!h->fused) {             // the quad sweep's second fields stay
        release(h->V_alt);
        release(h->I_alt);
    }
    for (float*& f : h->flux_alt) release(f);
}

static hipError_t device_malloc(ems_engine* h, void** q, size_t bytes)
{
    for (;;) {
        const hipError_t e = h->room(bytes) ? hipMalloc(q, bytes) : hipErrorOutOfMemory;
        if (e == hipSuccess) return e;
        (void)hipGetLastError();
        if (h->drop_read_buf()) continue;
        if (!h->pair) return e;
        leave_pairs(h);
    }
}

// the next one or two of at most `left` timesteps, and their samples: two in
// one launch where nothing samples the state between them; ev: the events of
// the step's (or, for a pair, its first step's) kernels; ahead: see launch_step
static int advance(ems_engine* h, unsigned left, hipEvent_t* ev, unsigned* done, bool& ahead)
{
    int rc;
    bool two = h->pair && left >= 2 && !probe_due(h, h->numTS + 1);
    for (size_t k = 0; k < h->dumps.size() && two; ++k) {
        unsigned ks;
        two = !dump_sample(h->dumps[k], h->numTS + 1, &ks);
    }
    *done = two ? 2 : 1;
    if (two) {
        PairBufs B{h->V, h->I, h->pmlV.flux_in, h->pmlI.flux_in, h->V_alt, h->I_alt, h->flux_alt[0], h->flux_alt[1],
                   h->numts_dev, h->numts_alt};
        void* args[] = {&h->pargs, &B};
        if (ev) (void)hipEventRecord(ev[0], h->stream);
        HIPCHK(hipLaunchKernel(pair_kernel(h, h->pair_lds > kPairLds * sizeof(float) * h->pair_threads), dim3(h->pair_blocks),
                               dim3(h->pair_threads), args, h->pair_lds, h->stream));
        if (ev) (void)hipEventRecord(ev[1], h->stream);
        swap_pair_buffers(h);
        ++h->pair_launches;
    } else if ((rc = launch_step(h, ev, left > 1, ahead))) return rc;
    h->numTS += *done;
    return launch_samples(h);
}

int ems_set_profiling(ems_engine* h, int enable)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    h->profile = enable != 0;
    return 0;
}

// steps of one ems_iterate call whose kernels are bracketed by events
constexpr unsigned kProfSteps = 4096;

// Steps per captured chunk: the requested length rounded up to a multiple of
// the period of the launch pattern (the sampling intervals of probes and
// dumps, the steady-state period, 2 for the buffer parity of a single-sweep
// form) when that period is at most 1024 steps, so that chunks repeat.
static unsigned graph_steps(const ems_engine* h)
{
    unsigned long long P = h->fused ? 2 : 1;
    auto add = [&P](unsigned v) {
        if (v) P = P / std::gcd(P, (unsigned long long)v) * v;
    };
    for (const auto& p : h->probes) {
        add(p.interval);
        add(p.fd_interval);
    }
    for (const auto& d : h->dumps) add(d.fd_interval);
    if (h->has_ss) add(h->ss.p);
    const unsigned c = h->graph_chunk;
    if (P > 1024) return c;
    return (unsigned)((c + P - 1) / P * P);
}

// launch pattern of the next `steps` steps from the host timestep on
static std::vector<unsigned char> chunk_key(const ems_engine* h, unsigned steps)
{
    std::vector<unsigned char> key;
    key.push_back((unsigned char)(((h->fused || h->pair) && h->V != h->V_base ? 1 : 0) |
                                  (h->pair && h->numts_dev > h->numts_alt ? 2 : 0)));
    for (unsigned k = 0; k < steps; ++k) {
        const unsigned ts = h->numTS + k;          // numTS before step k of the chunk
        unsigned char b = 0;
        if (h->has_ss && ts % h->ss.p == 0 && ts >= 2 * h->ss.p) b |= 1;
        if (!h->probes.empty() && probe_due(h, ts + 1)) b |= 2;
        key.push_back(b);
        for (size_t d = 0; d < h->dumps.size(); ++d) {
            unsigned ks;
            key.push_back((unsigned char)dump_sample(h->dumps[d], ts + 1, &ks));
        }
    }
    return key;
}

// one chunk of graph_chunk steps: replay the graph of its launch pattern,
// captured from the direct launches the first time the pattern occurs
static int graph_chunk(ems_engine* h, unsigned steps)
{
    // liveness of what the captured launches reference: every buffer a graph
    // names is an allocation of this engine, kept until ems_destroy; one made
    // after a capture (a table uploaded again) means the graphs may name the
    // previous one, so they are captured anew
    if (!h->graphs.empty() && h->graphs.front().nalloc != h->allocs.size()) drop_graphs(h);
    const std::vector<unsigned char> key = chunk_key(h, steps);
    ems_engine::GraphEnt* G = nullptr;
    for (auto& e : h->graphs)
        if (e.key == key) G = &e;
    if (G) {
        HIPCHK(hipGraphLaunch(G->exec, h->stream));
        // host state as the captured launches left it
        for (unsigned k = 2 * G->pairs; k < steps && h->fused; ++k) swap_step_buffers(h);
        if (G->pairs & 1u) swap_pair_buffers(h);
        h->pair_launches += G->pairs;
        h->numTS += steps;
        ++h->graph_replays;
        return 0;
    }
    if (h->graphs.size() >= kMaxGraphs) {
        // too many distinct patterns: direct launches
        bool ahead = false;
        for (unsigned k = 0, n; k < steps; k += n) {
            int rc = advance(h, steps - k, nullptr, &n, ahead);
            if (rc) return rc;
        }
        return 0;
    }
    ems_engine::GraphEnt e;
    e.key = key;
    HIPCHK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    int lrc = 0;
    const unsigned pairs0 = h->pair_launches;
    bool ahead = false;
    for (unsigned k = 0, n; k < steps && !lrc; k += n) lrc = advance(h, steps - k, nullptr, &n, ahead);
    e.pairs = h->pair_launches - pairs0;
    const hipError_t ec = hipStreamEndCapture(h->stream, &e.graph);
    if (lrc) {
        if (ec == hipSuccess && e.graph) (void)hipGraphDestroy(e.graph);
        return lrc;
    }
    if (ec != hipSuccess) return fail(EMS_E_HIP, std::string("graph capture failed: ") + hipGetErrorString(ec));
    HIPCHK(hipGraphInstantiate(&e.exec, e.graph, nullptr, nullptr, 0));
    HIPCHK(hipGraphLaunch(e.exec, h->stream));
    e.nalloc = h->allocs.size();
    h->graphs.push_back(std::move(e));
    ++h->graph_captures;
    return 0;
}

static void drop_graphs(ems_engine* h)
{
    if (!h->graphs.empty()) hipStreamSynchronize(h->stream);
    for (auto& G : h->graphs) {
        if (G.exec) hipGraphExecDestroy(G.exec);
        if (G.graph) hipGraphDestroy(G.graph);
    }
    h->graphs.clear();
}

int ems_set_graph(ems_engine* h, unsigned chunk_steps)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (chunk_steps > 4096) return fail(EMS_E_ARG, "graph chunk above 4096 steps");
    drop_graphs(h);
    h->graph_chunk = chunk_steps;
    return 0;
}

int ems_get_graph(const ems_engine* h, unsigned* chunk_steps, unsigned* captures, unsigned* replays)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (chunk_steps) *chunk_steps = h->graph_chunk;
    if (captures) *captures = h->graph_captures;
    if (replays) *replays = h->graph_replays;
    return 0;
}

int ems_iterate(ems_engine* h, unsigned nsteps)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    TxRange tx("ems_iterate");
    int rc;
    if (!h->inited && (rc = ems_init(h))) return rc;
    HIPCHK(hipSetDevice(h->device));
    rc = sync_probe_tables(h);
    if (rc) return rc;
    const unsigned nprof = h->profile ? std::min(nsteps, kProfSteps) : 0;
    while (h->kev.size() < 4 * (size_t)nprof) {
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        h->kev.push_back(e);
    }
    if (h->numTS == 0 && nsteps > 0) {
        // Process() before the first step (openems.cpp:1424-1425)
        if ((rc = launch_samples(h))) return rc;
        h->sampled0 = true;
    }
    HIPCHK(hipEventRecord(h->ev0, h->stream));
    unsigned s = 0;
    bool ahead = false;                   // false after each loop: its last step takes nothing along
    // step of the events' first four, and whether that launch held two steps
    std::vector<unsigned char> pairs(nprof, 0);
    for (unsigned n; s < nprof; s += n) {
        if ((rc = advance(h, nprof - s, &h->kev[4 * (size_t)s], &n, ahead))) return rc;
        pairs[s] = n == 2;
    }
    if (h->graph_chunk) {
        const unsigned steps = graph_steps(h);
        if (steps != h->graph_len) {
            drop_graphs(h);
            h->graph_len = steps;
        }
        while (nsteps - s >= steps) {
            TxRange txc("ems_iterate chunk");
            if ((rc = graph_chunk(h, steps))) return rc;
            s += steps;
        }
    }
    for (unsigned n; s < nsteps; s += n)
        if ((rc = advance(h, nsteps - s, nullptr, &n, ahead))) return rc;
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(h->ev1, h->stream));
    if (!h->async || nprof) {
        HIPCHK(hipEventSynchronize(h->ev1));
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, h->ev0, h->ev1));
        h->last_ms = ms;
    }
    if (nprof) {
        double vsum = 0, csum = 0, psum = 0;
        unsigned np = 0;
        for (unsigned s = 0; s < nprof; ++s) {
            float a = 0, b = 0;
            HIPCHK(hipEventElapsedTime(&a, h->kev[4 * (size_t)s], h->kev[4 * (size_t)s + 1]));
            if (pairs[s]) {
                psum += a;
                ++np;
                ++s;
                continue;
            }
            vsum += a;
            HIPCHK(hipEventElapsedTime(&b, h->kev[4 * (size_t)s + 2], h->kev[4 * (size_t)s + 3]));
            csum += b;
        }
        // with pairs: their launches' average, and no current half step beside them
        const unsigned one = nprof - 2 * np;
        h->last_volt_ms = np ? psum / np : vsum / one;
        h->last_curr_ms = np ? 0.0 : csum / one;
    }
    return 0;
}

unsigned ems_get_numts(const ems_engine* h) { return h ? h->numTS : 0; }

int ems_set_async(ems_engine* h, int async)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    h->async = async != 0;
    return 0;
}

int ems_sync(ems_engine* h)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    return 0;
}

constexpr size_t kReadBytes = 64u << 20;      // device buffer of a field read-out

// a field through host memory, a component at a time
static int get_field_staged(const ems_engine* h, const float* d, float* out)
{
    const unsigned* N = h->N;
    const size_t Nx = N[0], Ny = N[1], Nz = N[2];
    std::vector<float> stage(Nx * Ny * Nz);
    for (unsigned c = 0; c < 3; ++c) {
        HIPCHK(hipMemcpy(stage.data(), d + c * h->cs, stage.size() * sizeof(float), hipMemcpyDeviceToHost));
        parallel_rows(Nx * Ny, [&](size_t a, size_t b) {
            for (size_t r = a; r < b; ++r) {
                const float* q = stage.data() + r / Ny + Nx * (r % Ny);
                float* o = out + (c * Nx * Ny + r) * Nz;
                for (size_t z = 0; z < Nz; ++z) o[z] = q[z * Nx * Ny];
            }
        });
    }
    return 0;
}

static int get_field(ems_engine* h, const float* d, float* out)
{
    if (!h || !out) return fail(EMS_E_ARG, "null argument");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    // turned on the device, kReadBytes at a time; several threads may read at once
    std::lock_guard<std::mutex> lk(h->read_mu);
    const unsigned *N = h->N;
    const size_t row = (size_t)N[1] * N[2], rows = 3 * (size_t)N[0];     // floats of one x plane, planes of all components
    if (!h->read_buf) {
        // as many planes as the device has room for; with none, through the host
        size_t n = std::min(rows, std::max<size_t>(1, kReadBytes / (row * sizeof(float))));
        for (; n; n /= 2) {
            if (h->room(n * row * sizeof(float)) &&
                hipMalloc((void**)&h->read_buf, n * row * sizeof(float)) == hipSuccess) break;
            (void)hipGetLastError();
            h->read_buf = nullptr;
        }
        if (!n) return get_field_staged(h, d, out);
        h->read_rows = n;
        h->alloc_bytes += n * row * sizeof(float);
    }
    for (size_t r0 = 0; r0 < rows; r0 += h->read_rows) {
        const size_t r1 = std::min(rows, r0 + h->read_rows);
        for (size_t r = r0; r < r1;) {
            const unsigned c = (unsigned)(r / N[0]), x0 = (unsigned)(r % N[0]);
            const unsigned nx = (unsigned)std::min<size_t>(N[0] - x0, r1 - r);
            hipLaunchKernelGGL(k_to_nijk, dim3((nx + kTurn - 1) / kTurn, (N[2] + kTurn - 1) / kTurn, std::min(N[1], 65535u)),
                               dim3(kTurn * 8), 0, h->stream, d + c * h->cs, h->read_buf + (r - r0) * row, N[0], N[1], N[2],
                               x0, nx);
            r += nx;
        }
        HIPCHK(hipGetLastError());
        // a copy on the engine's own stream would set up staging of its own
        // first (the first read-out of a program 6.8 ms instead of 0.2)
        HIPCHK(hipStreamSynchronize(h->stream));
        HIPCHK(hipMemcpy(out + r0 * row, h->read_buf, (r1 - r0) * row * sizeof(float), hipMemcpyDeviceToHost));
    }
    return 0;
}

static int set_field(ems_engine* h, float* d, float* alt, const float* in)
{
    if (!h || !in) return fail(EMS_E_ARG, "null argument");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    int rc = upload_nijk(h, d, in);
    if (rc || !alt) return rc;
    // the fused step's second buffer must agree on the cells a step leaves alone
    // (a pair of timesteps leaves none alone)
    HIPCHK(hipMemcpy(alt, d, 3 * h->cs * sizeof(float), hipMemcpyDeviceToDevice));
    HIPCHK(hipDeviceSynchronize());
    return 0;
}

int ems_get_volt(ems_engine* h, float* out) { return h ? get_field(h, h->V, out) : fail(EMS_E_ARG, "null handle"); }
int ems_get_curr(ems_engine* h, float* out) { return h ? get_field(h, h->I, out) : fail(EMS_E_ARG, "null handle"); }
int ems_set_volt(ems_engine* h, const float* in)
{
    return h ? set_field(h, h->V, h->fused ? h->V_alt : nullptr, in) : fail(EMS_E_ARG, "null handle");
}
int ems_set_curr(ems_engine* h, const float* in)
{
    return h ? set_field(h, h->I, h->fused ? h->I_alt : nullptr, in) : fail(EMS_E_ARG, "null handle");
}

// one component's box [s, s+n) as x-fastest planes, through pitched copies
// of the device rows (dir: hipMemcpyDeviceToHost or HostToDevice)
static int box_copy(ems_engine* h, float* dev, float* host_xfast, const unsigned s[3], const unsigned n[3],
                    hipMemcpyKind dir)
{
    const size_t Nx = h->N[0], Ny = h->N[1];
    for (unsigned z = 0; z < n[2]; ++z) {
        float* d = dev + s[0] + Nx * (s[1] + Ny * (size_t)(s[2] + z));
        float* q = host_xfast + (size_t)z * n[0] * n[1];
        if (dir == hipMemcpyDeviceToHost)
            HIPCHK(hipMemcpy2D(q, n[0] * sizeof(float), d, Nx * sizeof(float), n[0] * sizeof(float), n[1], dir));
        else
            HIPCHK(hipMemcpy2D(d, Nx * sizeof(float), q, n[0] * sizeof(float), n[0] * sizeof(float), n[1], dir));
    }
    return 0;
}

static int box_check(const ems_engine* h, int comp, const unsigned start[3], const unsigned stop[3], unsigned n[3])
{
    if (comp < -1 || comp > 2) return fail(EMS_E_ARG, "field component must be 0, 1, 2 or -1 (all three)");
    for (int a = 0; a < 3; ++a) {
        if (start[a] > stop[a] || stop[a] >= h->N[a]) return fail(EMS_E_ARG, "field box outside the mesh");
        n[a] = stop[a] - start[a] + 1;
    }
    return 0;
}

int ems_read_field(ems_engine* h, int is_curr, int comp, const unsigned start[3], const unsigned stop[3], float* out)
{
    if (!h || !start || !stop || !out) return fail(EMS_E_ARG, "null argument");
    unsigned n[3];
    int rc = box_check(h, comp, start, stop, n);
    if (rc) return rc;
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    const size_t cnt = (size_t)n[0] * n[1] * n[2];
    std::vector<float> stage(cnt);
    const int c0 = comp < 0 ? 0 : comp, c1 = comp < 0 ? 2 : comp;
    float* F = is_curr ? h->I : h->V;
    for (int c = c0; c <= c1; ++c) {
        if ((rc = box_copy(h, F + (size_t)c * h->cs, stage.data(), start, n, hipMemcpyDeviceToHost))) return rc;
        float* o = out + (size_t)(c - c0) * cnt;
        for (unsigned x = 0; x < n[0]; ++x)
            for (unsigned y = 0; y < n[1]; ++y)
                for (unsigned z = 0; z < n[2]; ++z)
                    o[((size_t)x * n[1] + y) * n[2] + z] = stage[x + (size_t)n[0] * (y + (size_t)n[1] * z)];
    }
    return 0;
}

int ems_write_field(ems_engine* h, int is_curr, int comp, const unsigned start[3], const unsigned stop[3],
                    const float* in)
{
    if (!h || !start || !stop || !in) return fail(EMS_E_ARG, "null argument");
    unsigned n[3];
    int rc = box_check(h, comp, start, stop, n);
    if (rc) return rc;
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    const size_t cnt = (size_t)n[0] * n[1] * n[2];
    std::vector<float> stage(cnt);
    const int c0 = comp < 0 ? 0 : comp, c1 = comp < 0 ? 2 : comp;
    // the fused step's second buffer must agree on the cells a step leaves alone
    float* bufs[2] = {is_curr ? h->I : h->V, !h->fused ? nullptr : is_curr ? h->I_alt : h->V_alt};
    for (int c = c0; c <= c1; ++c) {
        const float* src = in + (size_t)(c - c0) * cnt;
        for (unsigned x = 0; x < n[0]; ++x)
            for (unsigned y = 0; y < n[1]; ++y)
                for (unsigned z = 0; z < n[2]; ++z)
                    stage[x + (size_t)n[0] * (y + (size_t)n[1] * z)] = src[((size_t)x * n[1] + y) * n[2] + z];
        for (float* F : bufs)
            if (F && (rc = box_copy(h, F + (size_t)c * h->cs, stage.data(), start, n, hipMemcpyHostToDevice))) return rc;
    }
    return 0;
}

int ems_get_field_at(ems_engine* h, int field, int interp, const unsigned pos[3], const double* const edge_len[3],
                     double out[3])
{
    if (!h || !pos || !edge_len || !out) return fail(EMS_E_ARG, "null argument");
    if (field != 0 && field != 1) return fail(EMS_E_ARG, "field must be 0 (E) or 1 (H)");
    if (interp < 0 || interp > 2) return fail(EMS_E_ARG, "interpolation must be 0 (none), 1 (node) or 2 (cell)");
    unsigned lo[3], hi[3], n[3];
    for (int a = 0; a < 3; ++a) {
        if (pos[a] >= h->N[a]) return fail(EMS_E_ARG, "position outside the mesh");
        if (!edge_len[a]) return fail(EMS_E_ARG, "null edge lengths");
        lo[a] = pos[a] ? pos[a] - 1 : 0;
        hi[a] = std::min(pos[a] + 1, h->N[a] - 1);
        n[a] = hi[a] - lo[a] + 1;
    }
    std::vector<float> box(3 * (size_t)n[0] * n[1] * n[2]);
    int rc = ems_read_field(h, field, -1, lo, hi, box.data());
    if (rc) return rc;
    for (int c = 0; c < 3; ++c) {
        const float* C = box.data() + (size_t)c * n[0] * n[1] * n[2];
        auto raw = [&](int dx, int dy, int dz) -> float {
            const unsigned x = pos[0] + dx - lo[0], y = pos[1] + dy - lo[1], z = pos[2] + dz - lo[2];
            return C[((size_t)x * n[1] + y) * n[2] + z];
        };
        out[c] = interp_value(field, interp, h->N, edge_len[c], pos, c, raw);
    }
    return 0;
}

int ems_energy(ems_engine* h, double* out)
{
    if (!h || !out) return fail(EMS_E_ARG, "null argument");
    HIPCHK(hipSetDevice(h->device));
    const unsigned nb = kEnergyBlocks;
    if (!h->energy_part) {           // before ems_init
        int rc = h->alloc(&h->energy_part, 2 * nb);
        if (rc) return rc;
    }
    double* part = h->energy_part;
    hipLaunchKernelGGL(k_energy, dim3(nb), dim3(kBlock), 0, h->stream, h->V, h->I, h->cs, h->N[0], h->N[1], h->N[2], part);
    std::vector<double> hp(2 * nb);
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipMemcpy(hp.data(), part, hp.size() * sizeof(double), hipMemcpyDeviceToHost));
    double e = 0, m = 0;
    for (unsigned b = 0; b < nb; ++b) {
        e += hp[2 * b];
        m += hp[2 * b + 1];
    }
    *out = 8.85418781762e-12 * e + 1.256637062e-6 * m;
    return 0;
}

// ems_energy without allocation or synchronisation: the partial sums go to
// the device's file-scope scratch, the result to the caller's device memory
int ems_energy_noalloc(ems_engine* h, double* d_out)
{
    if (!h || !d_out) return fail(EMS_E_ARG, "null argument");
    if (h->device < 0 || h->device >= kMaxDevices || !g_scratch_ptr[h->device])
        return fail(EMS_E_STATE, "the device scratch of this engine's device is not set up");
    HIPCHK(hipSetDevice(h->device));
    double* part = g_scratch_ptr[h->device];
    hipLaunchKernelGGL(k_energy, dim3(kEnergyBlocks), dim3(kBlock), 0, h->stream, h->V, h->I, h->cs, h->N[0], h->N[1],
                       h->N[2], part);
    hipLaunchKernelGGL(k_energy_total, dim3(1), dim3(64), 0, h->stream, part, kEnergyBlocks, d_out);
    HIPCHK(hipGetLastError());
    return 0;
}

int ems_last_timing(ems_engine* h, double* total_ms, double* volt_ms, double* curr_ms)
{
    if (!h) return fail(EMS_E_ARG, "null handle");
    if (total_ms) *total_ms = h->last_ms;
    if (volt_ms) *volt_ms = h->last_volt_ms;
    if (curr_ms) *curr_ms = h->last_curr_ms;
    return 0;
}

void ems_destroy(ems_engine* h)
{
    if (!h) return;
    hipSetDevice(h->device);
    if (h->stream) hipStreamSynchronize(h->stream);
    for (auto& G : h->graphs) {
        if (G.exec) hipGraphExecDestroy(G.exec);
        if (G.graph) hipGraphDestroy(G.graph);
    }
    for (const auto& a : h->allocs) hipFree(a.p);
    if (h->read_buf) hipFree(h->read_buf);
    if (h->ev0) hipEventDestroy(h->ev0);
    if (h->ev1) hipEventDestroy(h->ev1);
    for (auto& e : h->kev) hipEventDestroy(e);
    if (h->stream) hipStreamDestroy(h->stream);
    delete h;
}


// ---------------------------------------------------------------------------
// batched engine
// ---------------------------------------------------------------------------
}  // extern "C"

struct ems_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<ems_engine*> eng;
    int pm = kNoPml;
    bool cmp = false;
    std::vector<BatchInst> h_inst;
    BatchInst* d_inst = nullptr;
    // voltage sources in the voltage half step (every instance has its
    // lists); their tile masks hold for linear tiles only
    bool vsrc = false;
    std::vector<const unsigned*> vmask;
    // per-instance host lists, assembled into per-group device tables
    std::vector<std::vector<BatchExcGroup>> igrp[2];   // beg/end local to the instance's amp list
    std::vector<std::vector<float>> iamp[2];
    std::vector<std::vector<unsigned>> idel[2];
    std::vector<std::vector<BatchProbe>> iprobes;
    std::vector<size_t> ibytes;                         // device working set of each instance
    // groups of instances stepped together (all steps of a group run before
    // the next group starts, so a group that fits the last-level cache stays
    // resident); every group has its own work table and source / probe lists
    struct Group {
        std::vector<unsigned> inst;
        uint2* d_items = nullptr;
        unsigned nitems = 0, grid = 0;
        BatchExcGroup* d_grp[2] = {nullptr, nullptr};
        float* d_amp[2] = {nullptr, nullptr};
        unsigned* d_delay[2] = {nullptr, nullptr};
        unsigned G[2] = {0, 0};
        BatchProbe* d_probes = nullptr;
        unsigned nprobes = 0;
    };
    std::vector<Group> groups;
    std::vector<void*> gallocs;                         // group tables of the current configuration
    // each group's launches of graph_steps steps, captured once as a HIP graph
    // and replayed (0: direct launches, the default: replays measured no
    // faster on the batch, whose launches are long enough to hide the
    // launch overhead); dropped when the configuration changes
    unsigned graph_steps = 0;
    std::vector<hipGraphExec_t> gexec;
    // groups run on nstreams streams (group i on stream i % nstreams), so the
    // short source / probe launches and the last waves of one group's half
    // step overlap another group's work; stream 0 is `stream`
    unsigned nstreams = 1;
    std::vector<hipStream_t> xs;
    hipEvent_t fork = nullptr;
    std::vector<hipEvent_t> joins;
    hipStream_t gstream(size_t gi) const { return gi % nstreams == 0 ? stream : xs[gi % nstreams - 1]; }
    unsigned tx = 0, grid_req = 0;
    size_t group_bytes = 0;
    std::vector<unsigned> zdepth;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0;
    int resident = 0;                                    // workgroups resident per CU (occupancy)
    int cus = 0;
    std::vector<void*> allocs;

    template <typename T>
    int alloc(T** p, size_t n)
    {
        void* q = nullptr;
        hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
        if (e != hipSuccess) return fail(EMS_E_NOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
        allocs.push_back(q);
        *p = (T*)q;
        return 0;
    }
    template <typename T>
    int gupload(T** d, const T* src, size_t n)
    {
        void* q = nullptr;
        hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
        if (e != hipSuccess) return fail(EMS_E_NOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
        gallocs.push_back(q);
        *d = (T*)q;
        if (n) HIPCHK(hipMemcpy(q, src, n * sizeof(T), hipMemcpyHostToDevice));
        return 0;
    }
};

namespace {

template <int PM, bool CC, bool CURR>
void batch_launch_t(ems_batch* b, const ems_batch::Group& g, hipStream_t st)
{
    hipLaunchKernelGGL((k_batch_half<PM, CC, CURR>), dim3(g.grid), dim3(kBlock), 0, st, b->d_inst, g.d_items,
                       g.nitems);
}

template <bool CURR>
void batch_launch(ems_batch* b, const ems_batch::Group& g, hipStream_t st)
{
    if (b->cmp) {
        if (b->pm == kPmlCompressed) batch_launch_t<kPmlCompressed, true, CURR>(b, g, st);
        else if (b->pm == kPmlPlain) batch_launch_t<kPmlPlain, true, CURR>(b, g, st);
        else batch_launch_t<kNoPml, true, CURR>(b, g, st);
    } else {
        if (b->pm == kPmlCompressed) batch_launch_t<kPmlCompressed, false, CURR>(b, g, st);
        else if (b->pm == kPmlPlain) batch_launch_t<kPmlPlain, false, CURR>(b, g, st);
        else batch_launch_t<kNoPml, false, CURR>(b, g, st);
    }
}

// Configuration: tile shape, z depth per instance, grid size, and the
// working-set budget of a group (0: all instances in one group).  Groups are
// packed first-fit by decreasing working set.
void batch_drop_graphs(ems_batch* b)
{
    for (auto& x : b->gexec)
        if (x) hipGraphExecDestroy(x);
    b->gexec.clear();
}

int batch_build(ems_batch* b, unsigned tx, const std::vector<unsigned>& zd, unsigned grid, size_t group_bytes)
{
    const size_t n = b->eng.size();
    HIPCHK(hipStreamSynchronize(b->stream));
    batch_drop_graphs(b);
    for (void* p : b->gallocs) hipFree(p);
    b->gallocs.clear();
    b->groups.clear();
    for (size_t i = 0; i < n; ++i) {
        BatchInst& B = b->h_inst[i];
        B.g.zdepth = zd[i];
        set_tiles(B.g, tx);
        if (b->vsrc) B.vsrc.tmask = tx == 0 ? b->vmask[i] : nullptr;
        if ((unsigned long long)B.g.qtiles * B.g.nzc > 0xFFFFFFFFull)
            return fail(EMS_E_ARG, "instance too large for the batch work table");
    }
    HIPCHK(hipMemcpy(b->d_inst, b->h_inst.data(), n * sizeof(BatchInst), hipMemcpyHostToDevice));
    // partition
    std::vector<std::vector<unsigned>> parts;
    if (group_bytes == 0) {
        parts.emplace_back();
        for (unsigned i = 0; i < n; ++i) parts[0].push_back(i);
    } else {
        std::vector<unsigned> order(n);
        for (unsigned i = 0; i < n; ++i) order[i] = i;
        std::stable_sort(order.begin(), order.end(), [&](unsigned a, unsigned c) { return b->ibytes[a] > b->ibytes[c]; });
        std::vector<size_t> load;
        for (unsigned i : order) {
            size_t k = 0;
            while (k < parts.size() && load[k] + b->ibytes[i] > group_bytes) ++k;
            if (k == parts.size()) {
                parts.emplace_back();
                load.push_back(0);
            }
            parts[k].push_back(i);
            load[k] += b->ibytes[i];
        }
        for (auto& p : parts) std::sort(p.begin(), p.end());
    }
    for (const auto& p : parts) {
        ems_batch::Group g;
        g.inst = p;
        std::vector<uint2> items;
        for (unsigned i : p) {
            const BatchInst& B = b->h_inst[i];
            const unsigned cnt = B.g.qtiles * B.g.nzc;
            for (unsigned t = 0; t < cnt; ++t) items.push_back(make_uint2(i, t));
        }
        int rc;
        if ((rc = b->gupload(&g.d_items, items.data(), items.size()))) return rc;
        g.nitems = (unsigned)items.size();
        g.grid = grid == 0 ? g.nitems : std::min(grid, g.nitems);
        for (int c = 0; c < 2; ++c) {
            std::vector<BatchExcGroup> grp;
            std::vector<float> amp;
            std::vector<unsigned> del;
            for (unsigned i : p) {
                for (BatchExcGroup q : b->igrp[c][i]) {
                    q.beg += (unsigned)amp.size();
                    q.end += (unsigned)amp.size();
                    grp.push_back(q);
                }
                amp.insert(amp.end(), b->iamp[c][i].begin(), b->iamp[c][i].end());
                del.insert(del.end(), b->idel[c][i].begin(), b->idel[c][i].end());
            }
            g.G[c] = (unsigned)grp.size();
            if (g.G[c] && ((rc = b->gupload(&g.d_grp[c], grp.data(), grp.size())) ||
                           (rc = b->gupload(&g.d_amp[c], amp.data(), amp.size())) ||
                           (rc = b->gupload(&g.d_delay[c], del.data(), del.size()))))
                return rc;
        }
        std::vector<BatchProbe> pr;
        for (unsigned i : p) pr.insert(pr.end(), b->iprobes[i].begin(), b->iprobes[i].end());
        g.nprobes = (unsigned)pr.size();
        if (g.nprobes && (rc = b->gupload(&g.d_probes, pr.data(), pr.size()))) return rc;
        b->groups.push_back(g);
    }
    b->tx = tx;
    b->zdepth = zd;
    b->grid_req = grid;
    b->group_bytes = group_bytes;
    return 0;
}

void batch_step(ems_batch* b, const ems_batch::Group& g, hipStream_t st)
{
    const unsigned T = 256;
    batch_launch<false>(b, g, st);
    if (g.G[0] && !b->vsrc)
        hipLaunchKernelGGL(k_batch_excite, dim3((g.G[0] + T - 1) / T), dim3(T), 0, st, b->d_inst, g.d_grp[0],
                           g.G[0], g.d_amp[0], g.d_delay[0], 0, 0);
    batch_launch<true>(b, g, st);
    if (g.G[1])
        hipLaunchKernelGGL(k_batch_excite, dim3((g.G[1] + T - 1) / T), dim3(T), 0, st, b->d_inst, g.d_grp[1],
                           g.G[1], g.d_amp[1], g.d_delay[1], 1, -1);
    if (g.nprobes)
        hipLaunchKernelGGL(k_batch_probe, dim3(g.nprobes), dim3(kBlock), 0, st, b->d_inst, g.d_probes);
}

// All kernel arguments of a step are the same at every step (the timestep
// is read on the device), so a chunk of steps replays as a graph.
int batch_run(ems_batch* b, unsigned nsteps)
{
    const unsigned S = b->graph_steps;
    if (S && b->gexec.size() != b->groups.size()) b->gexec.assign(b->groups.size(), nullptr);
    if (b->nstreams > 1) {
        // fork: the other streams start after what is queued on stream 0
        HIPCHK(hipEventRecord(b->fork, b->stream));
        for (auto st : b->xs) HIPCHK(hipStreamWaitEvent(st, b->fork, 0));
    }
    for (size_t gi = 0; gi < b->groups.size(); ++gi) {
        const auto& g = b->groups[gi];
        hipStream_t st = b->gstream(gi);
        unsigned s = 0;
        if (S && nsteps >= S) {
            if (!b->gexec[gi]) {
                hipGraph_t graph;
                HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
                for (unsigned k = 0; k < S; ++k) batch_step(b, g, st);
                HIPCHK(hipStreamEndCapture(st, &graph));
                hipError_t e = hipGraphInstantiate(&b->gexec[gi], graph, nullptr, nullptr, 0);
                hipGraphDestroy(graph);
                if (e != hipSuccess) {
                    b->gexec[gi] = nullptr;
                    return fail(EMS_E_HIP, std::string("graph instantiation failed: ") + hipGetErrorString(e));
                }
            }
            for (; s + S <= nsteps; s += S) HIPCHK(hipGraphLaunch(b->gexec[gi], st));
        }
        for (; s < nsteps; ++s) batch_step(b, g, st);
    }
    if (b->nstreams > 1)
        // join: stream 0 continues after every other stream's work
        for (size_t k = 0; k < b->xs.size(); ++k) {
            HIPCHK(hipEventRecord(b->joins[k], b->xs[k]));
            HIPCHK(hipStreamWaitEvent(b->stream, b->joins[k], 0));
        }
    return 0;
}

}  // namespace

extern "C" {

int ems_batch_create(ems_batch** out, ems_engine* const* engines, unsigned count)
{
    if (!out || !engines || count == 0) return fail(EMS_E_ARG, "null argument or empty batch");
    *out = nullptr;
    const ems_engine* e0 = engines[0];
    if (!e0) return fail(EMS_E_ARG, "null engine");
    for (unsigned i = 0; i < count; ++i) {
        const ems_engine* e = engines[i];
        if (!e) return fail(EMS_E_ARG, "null engine");
        if (!e->inited) return fail(EMS_E_STATE, "batch engines must be initialised (ems_init)");
        if (e->device != e0->device) return fail(EMS_E_ARG, "batch engines must share one device");
        if (e->cmp != e0->cmp) return fail(EMS_E_ARG, "batch engines must share one coefficient layout");
        const int pm = e->pmlV.n ? e->pml_mode : kNoPml, pm0 = e0->pmlV.n ? e0->pml_mode : kNoPml;
        if (pm != pm0) return fail(EMS_E_ARG, "batch engines must share one UPML layout (all with or all without)");
        if (!e->mur.empty() || !e->lor.empty() || !e->rlc.empty() || !e->dumps.empty() || e->has_ss)
            return fail(EMS_E_ARG, "batched instances support UPML, sources and probes only");
        if (e->fused) return fail(EMS_E_ARG, "batched instances run two half steps (ems_set_fused(h, 0))");
        if (e->numTS != e0->numTS) return fail(EMS_E_STATE, "batch engines must be at the same timestep");
        for (unsigned j = 0; j < i; ++j)
            if (engines[j] == e) return fail(EMS_E_ARG, "an engine appears twice in the batch");
    }
    HIPCHK(hipSetDevice(e0->device));
    // an instance names its engine's field, flux and counter buffers for good:
    // an engine that went on advancing in pairs by itself would swap them
    for (unsigned i = 0; i < count; ++i) leave_pairs(engines[i]);
    ems_batch* b = new ems_batch();
    auto bail = [&](int r) {
        ems_batch_destroy(b);
        return r;
    };
    b->device = e0->device;
    b->eng.assign(engines, engines + count);
    b->cmp = e0->cmp;
    b->pm = e0->pmlV.n ? e0->pml_mode : kNoPml;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(EMS_E_HIP, "stream creation failed"));
    hipEventCreate(&b->ev0);
    hipEventCreate(&b->ev1);
    int rc;
    for (int c = 0; c < 2; ++c) {
        b->igrp[c].resize(count);
        b->iamp[c].resize(count);
        b->idel[c].resize(count);
    }
    b->iprobes.resize(count);
    for (unsigned i = 0; i < count; ++i) {
        ems_engine* e = engines[i];
        HIPCHK(hipStreamSynchronize(e->stream));
        if ((rc = sync_probe_tables(e))) return bail(rc);
        BatchInst B{};
        B.g = e->g;
        B.V = e->V;
        B.I = e->I;
        B.kV = e->kV;
        B.kI = e->kI;
        B.pV = e->pmlV;
        B.pI = e->pmlI;
        B.numts = e->numts_dev;
        B.sig[0] = e->sig[0];
        B.sig[1] = e->sig[1];
        B.sigLen = e->sigLen;
        B.period = e->period;
        B.vsrc = e->quad ? ExcArgs{} : e->qsrc;
        b->h_inst.push_back(B);
        b->zdepth.push_back(e->g.zdepth);
        // device working set: fields, coefficients, UPML
        size_t bytes = 2 * 3 * e->cs * sizeof(float);
        bytes += e->cmp ? e->cs * sizeof(unsigned short) + 2 * 32 * (size_t)e->n_unique : 4 * 3 * e->cs * sizeof(float);
        if (e->pmlV.n) {
            const size_t np = e->pmlV.npos;
            bytes += 2 * 3 * np * sizeof(float);
            bytes += e->pml_mode == kPmlCompressed ? np * sizeof(unsigned) + 2 * 48 * (size_t)e->n_unique_pml
                                                   : 2 * 9 * np * sizeof(float);
        }
        b->ibytes.push_back(bytes);
        for (int c = 0; c < 2; ++c) {
            const auto& E = e->exc[c];
            for (unsigned g = 0; g < E.G; ++g) {
                BatchExcGroup q{};
                q.inst = i;
                q.lin = E.h_glin[g];
                q.beg = E.h_gbeg[g];
                q.end = E.h_gbeg[g + 1];
                b->igrp[c][i].push_back(q);
            }
            b->iamp[c][i] = E.h_amp;
            b->idel[c][i] = E.h_delay;
        }
        for (const auto& P : e->probes) {
            BatchProbe q{};
            q.P = P;
            q.inst = i;
            q.elin = e->d_elin;
            q.esign = e->d_esign;
            q.ediv = e->d_ediv;
            b->iprobes[i].push_back(q);
        }
    }
    b->vsrc = true;
    for (const auto& B : b->h_inst) b->vsrc = b->vsrc && B.vsrc.beg;
    for (auto& B : b->h_inst) {
        if (!b->vsrc) B.vsrc = ExcArgs{};
        b->vmask.push_back(B.vsrc.tmask);
    }
    if ((rc = b->alloc(&b->d_inst, count))) return bail(rc);
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, b->device));
    b->cus = prop.multiProcessorCount;
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_batch_half<kPmlCompressed, true, false>, kBlock, 0) !=
            hipSuccess ||
        occ <= 0)
        occ = 4;
    b->resident = occ;
    // default: each instance's own depth, linear tiles, one workgroup per item, one group
    if ((rc = batch_build(b, 0, b->zdepth, 0, 0))) return bail(rc);
    *out = b;
    return 0;
}

int ems_batch_set_config(ems_batch* b, unsigned tile_x, const unsigned* zdepth, unsigned grid)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (tile_x != 0 && (tile_x > kBlock || kBlock % tile_x || tile_x < 8))
        return fail(EMS_E_ARG, "tile_x must be 0 or a divisor of 256 from 8 to 256");
    std::vector<unsigned> zd(b->eng.size());
    for (size_t i = 0; i < zd.size(); ++i) {
        zd[i] = zdepth ? zdepth[i] : choose_zdepth(b->eng[i]->N);
        if (zd[i] < 1 || zd[i] > 4096) return fail(EMS_E_ARG, "z depth out of range");
    }
    return batch_build(b, tile_x, zd, grid, b->group_bytes);
}

int ems_batch_set_grouping(ems_batch* b, unsigned long long group_bytes)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    return batch_build(b, b->tx, b->zdepth, b->grid_req, (size_t)group_bytes);
}

int ems_batch_get_config(const ems_batch* b, unsigned* tile_x, unsigned* zdepth, unsigned* grid, unsigned* nitems)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (tile_x) *tile_x = b->tx;
    if (zdepth)
        for (size_t i = 0; i < b->zdepth.size(); ++i) zdepth[i] = b->zdepth[i];
    if (grid) *grid = b->grid_req;
    if (nitems) {
        unsigned t = 0;
        for (const auto& g : b->groups) t += g.nitems;
        *nitems = t;
    }
    return 0;
}

int ems_batch_get_grouping(const ems_batch* b, unsigned long long* group_bytes, unsigned* ngroups)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (group_bytes) *group_bytes = b->group_bytes;
    if (ngroups) *ngroups = (unsigned)b->groups.size();
    return 0;
}

int ems_batch_iterate(ems_batch* b, unsigned nsteps)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    TxRange tx("ems_batch_iterate");
    HIPCHK(hipSetDevice(b->device));
    for (auto* e : b->eng) HIPCHK(hipStreamSynchronize(e->stream));
    if (b->eng[0]->numTS == 0 && nsteps > 0)
        // Process() before the first step (openems.cpp:1424-1425)
        for (const auto& g : b->groups)
            if (g.nprobes)
                hipLaunchKernelGGL(k_batch_probe, dim3(g.nprobes), dim3(kBlock), 0, b->stream, b->d_inst, g.d_probes);
    HIPCHK(hipEventRecord(b->ev0, b->stream));
    int rc = batch_run(b, nsteps);
    if (rc) return rc;
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(b->ev1, b->stream));
    HIPCHK(hipEventSynchronize(b->ev1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    b->last_ms = ms;
    for (auto* e : b->eng) e->numTS += nsteps;
    return 0;
}

// Autotuner: time every candidate tile shape x z-depth policy x grid size x
// (stream count, group budget) on the batch itself for `steps` steps of all
// groups, restore the state the candidates advanced (fields, UPML fluxes,
// counters, probe sample counts), and keep the fastest.  Depth policies: each
// instance's own (choose_zdepth), 4 or 8 for all; grids: one workgroup per
// work item or the resident workgroups; plans: one stream with one group or
// budgets of 128-224 MiB, two streams with 80-112 MiB, three with 56-64 MiB
// (the last-level cache holds 256 MiB; the budget also sets how many work
// items a group's launches spread over the resident workgroups).
int ems_batch_autotune(ems_batch* b, unsigned steps, double* best_ms)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (steps < 2) steps = 2;
    HIPCHK(hipSetDevice(b->device));
    for (auto* e : b->eng) HIPCHK(hipStreamSynchronize(e->stream));
    struct Saved {
        float *V, *I, *fV, *fI;
        unsigned numts[2];
        std::vector<unsigned> counts;
    };
    std::vector<Saved> sv(b->eng.size());
    std::vector<void*> tmp;
    auto cleanup = [&]() {
        for (void* p : tmp) (void)hipFree(p);
    };
    auto dalloc = [&](float** p, size_t n) -> bool {
        void* q = nullptr;
        if (hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(float)) != hipSuccess) return false;
        tmp.push_back(q);
        *p = (float*)q;
        return true;
    };
    // every snapshot / restore copy is checked; the first failure is kept
    hipError_t cerr = hipSuccess;
    const char* cwhat = "";
    auto cp = [&](void* dst, const void* src, size_t bytes, hipMemcpyKind kind, const char* what) {
        const hipError_t e = hipMemcpy(dst, src, bytes, kind);
        if (e != hipSuccess && cerr == hipSuccess) {
            cerr = e;
            cwhat = what;
        }
    };
    auto copy_failed = [&](const char* phase) {
        return fail(EMS_E_HIP, std::string("ems_batch_autotune: ") + phase + " copy of " + cwhat + " failed: " +
                                   hipGetErrorString(cerr));
    };
    for (size_t i = 0; i < b->eng.size(); ++i) {
        ems_engine* e = b->eng[i];
        Saved& S = sv[i];
        S.fV = S.fI = nullptr;
        if (!dalloc(&S.V, 3 * e->cs) || !dalloc(&S.I, 3 * e->cs)) {
            cleanup();
            return fail(EMS_E_NOMEM, "no device memory for the autotuner's snapshot");
        }
        cp(S.V, e->V, 3 * e->cs * sizeof(float), hipMemcpyDeviceToDevice, "voltages");
        cp(S.I, e->I, 3 * e->cs * sizeof(float), hipMemcpyDeviceToDevice, "currents");
        if (e->pmlV.n) {
            if (!dalloc(&S.fV, 3 * e->pmlV.npos) || !dalloc(&S.fI, 3 * e->pmlI.npos)) {
                cleanup();
                return fail(EMS_E_NOMEM, "no device memory for the autotuner's snapshot");
            }
            cp(S.fV, e->pmlV.flux_in, 3 * e->pmlV.npos * sizeof(float), hipMemcpyDeviceToDevice, "voltage flux");
            cp(S.fI, e->pmlI.flux_in, 3 * e->pmlI.npos * sizeof(float), hipMemcpyDeviceToDevice, "current flux");
        }
        cp(S.numts, e->numts_dev, 2 * sizeof(unsigned), hipMemcpyDeviceToHost, "step counter");
        for (const auto& P : e->probes) {
            unsigned c = 0;
            cp(&c, P.count, sizeof(unsigned), hipMemcpyDeviceToHost, "probe count");
            S.counts.push_back(c);
        }
    }
    if (cerr != hipSuccess) {
        cleanup();
        return copy_failed("snapshot");
    }
    {
        const hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) {
            cleanup();
            return fail(EMS_E_HIP, std::string("ems_batch_autotune: ") + hipGetErrorString(e));
        }
    }
    // puts every instance back to the snapshot; returns 0 or an EMS_E_HIP
    // status (the instances are then in an undefined state)
    auto restore = [&]() -> int {
        for (size_t i = 0; i < b->eng.size(); ++i) {
            ems_engine* e = b->eng[i];
            Saved& S = sv[i];
            cp(e->V, S.V, 3 * e->cs * sizeof(float), hipMemcpyDeviceToDevice, "voltages");
            cp(e->I, S.I, 3 * e->cs * sizeof(float), hipMemcpyDeviceToDevice, "currents");
            if (e->pmlV.n) {
                cp(const_cast<float*>(e->pmlV.flux_in), S.fV, 3 * e->pmlV.npos * sizeof(float),
                   hipMemcpyDeviceToDevice, "voltage flux");
                cp(const_cast<float*>(e->pmlI.flux_in), S.fI, 3 * e->pmlI.npos * sizeof(float),
                   hipMemcpyDeviceToDevice, "current flux");
            }
            cp(e->numts_dev, S.numts, 2 * sizeof(unsigned), hipMemcpyHostToDevice, "step counter");
            for (size_t k = 0; k < e->probes.size(); ++k)
                cp(e->probes[k].count, &S.counts[k], sizeof(unsigned), hipMemcpyHostToDevice, "probe count");
        }
        // device-to-device copies are not ordered with the batch's stream
        const hipError_t se = hipDeviceSynchronize();
        if (se != hipSuccess && cerr == hipSuccess) {
            cerr = se;
            cwhat = "(synchronisation)";
        }
        return cerr == hipSuccess ? 0 : copy_failed("restore");
    };
    const unsigned txs[2] = {0, 64};
    const unsigned depths[3] = {0, 4, 8};   // 0: each instance's own choice
    const unsigned grids[2] = {0, (unsigned)(b->resident * b->cus)};
    const size_t mib = size_t(1) << 20;
    // (streams, group budget): one stream with budgets up to the cache size,
    // several streams with a budget near the cache size over the stream count
    const std::pair<unsigned, size_t> plans[] = {{1, 0},        {1, 128 * mib}, {1, 160 * mib}, {1, 192 * mib},
                                                 {1, 224 * mib}, {2, 80 * mib},  {2, 96 * mib},  {2, 112 * mib},
                                                 {3, 56 * mib},  {3, 64 * mib}};
    const unsigned streams0 = b->nstreams;
    double best = 1e30;
    unsigned btx = 0, bdep = 0, bgrid = 0, bns = streams0;
    size_t bbud = 0;
    for (const auto& plan : plans)
        for (unsigned tx : txs)
            for (unsigned dep : depths)
                for (unsigned grid : grids) {
                    std::vector<unsigned> zd(b->eng.size());
                    for (size_t i = 0; i < zd.size(); ++i) zd[i] = dep ? dep : choose_zdepth(b->eng[i]->N);
                    int rc = batch_build(b, tx, zd, grid, plan.second);
                    if (!rc) rc = ems_batch_set_streams(b, plan.first);
                    if (rc) {
                        const int rr = restore();
                        cleanup();
                        return rr ? rr : rc;
                    }
                    // one warm-up step of every group, then steps-1 timed steps of all groups
                    if ((rc = batch_run(b, 1))) {
                        const int rr = restore();
                        cleanup();
                        return rr ? rr : rc;
                    }
                    hipError_t te = hipEventRecord(b->ev0, b->stream);
                    rc = batch_run(b, steps - 1);
                    if (te == hipSuccess) te = hipEventRecord(b->ev1, b->stream);
                    if (te == hipSuccess) te = hipEventSynchronize(b->ev1);
                    float ms = 0;
                    if (te == hipSuccess) te = hipEventElapsedTime(&ms, b->ev0, b->ev1);
                    if (!rc && te != hipSuccess)
                        rc = fail(EMS_E_HIP, std::string("ems_batch_autotune: timing: ") + hipGetErrorString(te));
                    if (rc) {
                        const int rr = restore();
                        cleanup();
                        return rr ? rr : rc;
                    }
                    const double tot = ms / (steps - 1);
                    if (tot < best) {
                        best = tot;
                        btx = tx;
                        bdep = dep;
                        bgrid = grid;
                        bbud = plan.second;
                        bns = plan.first;
                    }
                    if ((rc = restore())) {
                        cleanup();
                        return rc;
                    }
                }
    std::vector<unsigned> zd(b->eng.size());
    for (size_t i = 0; i < zd.size(); ++i) zd[i] = bdep ? bdep : choose_zdepth(b->eng[i]->N);
    int rc = batch_build(b, btx, zd, bgrid, bbud);
    if (!rc) rc = ems_batch_set_streams(b, bns);
    const hipError_t se = hipStreamSynchronize(b->stream);
    cleanup();
    if (!rc && se != hipSuccess)
        rc = fail(EMS_E_HIP, std::string("ems_batch_autotune: ") + hipGetErrorString(se));
    if (best_ms) *best_ms = best;
    return rc;
}

int ems_batch_last_ms(const ems_batch* b, double* ms)
{
    if (!b || !ms) return fail(EMS_E_ARG, "null argument");
    *ms = b->last_ms;
    return 0;
}

int ems_batch_set_graph(ems_batch* b, unsigned steps)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (steps > 4096) return fail(EMS_E_ARG, "graph chunk longer than 4096 steps");
    HIPCHK(hipSetDevice(b->device));
    HIPCHK(hipStreamSynchronize(b->stream));
    batch_drop_graphs(b);
    b->graph_steps = steps;
    return 0;
}

int ems_batch_set_streams(ems_batch* b, unsigned n)
{
    if (!b) return fail(EMS_E_ARG, "null batch");
    if (n < 1 || n > 4) return fail(EMS_E_ARG, "stream count must be 1..4");
    HIPCHK(hipSetDevice(b->device));
    HIPCHK(hipStreamSynchronize(b->stream));
    for (auto st : b->xs) HIPCHK(hipStreamSynchronize(st));
    batch_drop_graphs(b);       // captured on the streams of the old assignment
    if (!b->fork) HIPCHK(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
    while (b->xs.size() < n - 1) {
        hipStream_t st;
        HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        b->xs.push_back(st);
        hipEvent_t ev;
        HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        b->joins.push_back(ev);
    }
    while (b->xs.size() > n - 1) {
        hipStreamDestroy(b->xs.back());
        hipEventDestroy(b->joins.back());
        b->xs.pop_back();
        b->joins.pop_back();
    }
    b->nstreams = n;
    return 0;
}

int ems_batch_get_streams(const ems_batch* b, unsigned* n)
{
    if (!b || !n) return fail(EMS_E_ARG, "null argument");
    *n = b->nstreams;
    return 0;
}

int ems_batch_get_graph(const ems_batch* b, unsigned* steps)
{
    if (!b || !steps) return fail(EMS_E_ARG, "null argument");
    *steps = b->graph_steps;
    return 0;
}

void ems_batch_destroy(ems_batch* b)
{
    if (!b) return;
    hipSetDevice(b->device);
    if (b->stream) hipStreamSynchronize(b->stream);
    for (auto st : b->xs) hipStreamSynchronize(st);
    batch_drop_graphs(b);
    for (auto st : b->xs) hipStreamDestroy(st);
    for (auto ev : b->joins) hipEventDestroy(ev);
    if (b->fork) hipEventDestroy(b->fork);
    for (void* p : b->gallocs) hipFree(p);
    for (void* p : b->allocs) hipFree(p);
    if (b->ev0) hipEventDestroy(b->ev0);
    if (b->ev1) hipEventDestroy(b->ev1);
    if (b->stream) hipStreamDestroy(b->stream);
    delete b;
}


// ---------------------------------------------------------------------------
// adjoint gradients
// ---------------------------------------------------------------------------
}  // extern "C"

namespace {

// one saved state: fields, UPML fluxes, timestep
struct AdjCkpt {
    float *V = nullptr, *I = nullptr, *FV = nullptr, *FI = nullptr;
    unsigned ts = 0;
};

}  // namespace

struct ems_adjoint {
    ems_engine* h = nullptr;
    AdjProbe* d_probes = nullptr;
    unsigned np = 0;
    double freq = 0, dT = 0;
    AdjBox box{};
    unsigned K = 256;
    unsigned n0 = 0, nsteps = 0;
    double* d_F = nullptr;
    std::vector<double> F;
    std::vector<AdjCkpt> ck;   // state at n0 + s*K, s = 0..S-1, then the final state
    float *lV = nullptr, *lI = nullptr, *A = nullptr, *B = nullptr, *lFV = nullptr, *lFI = nullptr;
    // recorded inputs of the voltage updates, [rec_steps][3][box.n] each: of
    // every forward step where they fit (kept), else of one segment
    float *hc = nullptr, *hv = nullptr;
    size_t rec_steps = 0;
    bool kept = false;
    double *gvi = nullptr, *gvv = nullptr;
    bool forward_done = false;
    std::vector<void*> allocs;
    template <typename T>
    int alloc(T** p, size_t n)
    {
        void* q = nullptr;
        hipError_t e = device_malloc(h, &q, std::max<size_t>(n, 1) * sizeof(T));
        if (e != hipSuccess) return fail(EMS_E_NOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
        allocs.push_back(q);
        *p = (T*)q;
        return 0;
    }
};

namespace {

int adj_save(ems_adjoint* a, AdjCkpt& c)
{
    ems_engine* h = a->h;
    const size_t fb = 3 * h->cs * sizeof(float);
    int rc;
    if (!c.V) {
        if ((rc = a->alloc(&c.V, 3 * h->cs)) || (rc = a->alloc(&c.I, 3 * h->cs))) return rc;
        if (h->pmlV.n && ((rc = a->alloc(&c.FV, 3 * h->pmlV.npos)) || (rc = a->alloc(&c.FI, 3 * h->pmlI.npos))))
            return rc;
    }
    HIPCHK(hipMemcpyAsync(c.V, h->V, fb, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(c.I, h->I, fb, hipMemcpyDeviceToDevice, h->stream));
    if (h->pmlV.n) {
        HIPCHK(hipMemcpyAsync(c.FV, h->pmlV.flux_in, 3 * h->pmlV.npos * sizeof(float), hipMemcpyDeviceToDevice,
                              h->stream));
        HIPCHK(hipMemcpyAsync(c.FI, h->pmlI.flux_in, 3 * h->pmlI.npos * sizeof(float), hipMemcpyDeviceToDevice,
                              h->stream));
    }
    c.ts = h->numTS;
    return 0;
}

int adj_restore(ems_adjoint* a, const AdjCkpt& c)
{
    ems_engine* h = a->h;
    const size_t fb = 3 * h->cs * sizeof(float);
    HIPCHK(hipMemcpyAsync(h->V, c.V, fb, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->I, c.I, fb, hipMemcpyDeviceToDevice, h->stream));
    if (h->pmlV.n) {
        HIPCHK(hipMemcpyAsync(const_cast<float*>(h->pmlV.flux_in), c.FV, 3 * h->pmlV.npos * sizeof(float),
                              hipMemcpyDeviceToDevice, h->stream));
        HIPCHK(hipMemcpyAsync(const_cast<float*>(h->pmlI.flux_in), c.FI, 3 * h->pmlI.npos * sizeof(float),
                              hipMemcpyDeviceToDevice, h->stream));
    }
    const unsigned ts[2] = {c.ts, 0u};
    HIPCHK(hipMemcpyAsync(h->numts_dev, ts, sizeof(ts), hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    h->numTS = c.ts;
    return 0;
}

// Records of every forward step, or of one segment.  Kept, they save the
// reverse pass its replay of the forward steps (a third of it): the box is a
// small part of the mesh (17 x 17 x 7 edges: 48 KB a step), so they stay
// wherever they take at most an eighth of the free memory; beyond that the
// states saved every K steps are replayed.  EMS_ADJ_KEEP=0 always replays.
int adj_reserve(ems_adjoint* a, unsigned nsteps)
{
    const size_t step = 3 * a->box.n * sizeof(float);
    auto release = [&] {
        if (a->hc) (void)hipFree(a->hc);
        if (a->hv) (void)hipFree(a->hv);
        a->hc = a->hv = nullptr;
        a->rec_steps = 0;
    };
    auto grow = [&](size_t n) {
        if (a->rec_steps >= n) return true;
        release();
        if (device_malloc(a->h, (void**)&a->hc, n * step) != hipSuccess ||
            device_malloc(a->h, (void**)&a->hv, n * step) != hipSuccess) {
            release();
            return false;
        }
        a->rec_steps = n;
        return true;
    };
    size_t freeb = 0, totalb = 0;
    bool keep = true;
    if (const char* e = std::getenv("EMS_ADJ_KEEP")) keep = std::atoi(e) != 0;
    if (a->rec_steps < nsteps)
        keep = keep && hipMemGetInfo(&freeb, &totalb) == hipSuccess && 2 * (unsigned long long)nsteps * step <= freeb / 8;
    a->kept = keep && grow(nsteps);
    if (!a->kept && !grow(std::min(a->K, nsteps))) return fail(EMS_E_NOMEM, "no device memory for the adjoint's records");
    return 0;
}

// the record of step `rec` (-1: none) and, after a forward step, the running DFT
void adj_sample(ems_adjoint* a, int rec, bool dft)
{
    ems_engine* h = a->h;
    const unsigned rblk = rec < 0 ? 0 : (unsigned)((a->box.n + kBlock - 1) / kBlock);
    const unsigned np = dft ? a->np : 0, nb = rblk + (np + kBlock - 1) / kBlock;
    const size_t at = rec < 0 ? 0 : (size_t)rec * 3 * a->box.n;
    if (nb)
        hipLaunchKernelGGL(k_adj_sample, dim3(nb), dim3(kBlock), 0, h->stream, h->g, h->V, h->I, a->box, a->hc + at,
                           a->hv + at, rblk, a->d_probes, np, a->freq, a->dT, h->numts_dev, a->d_F);
}

template <int PM, bool CC>
void adj_kernels_t(ems_adjoint* a, const float* hc, const float* hv, unsigned ts)
{
    ems_engine* h = a->h;
    const unsigned nblk = h->g.qtiles * h->g.nzc;
    PmlArgs pI = h->pmlI, pV = h->pmlV;
    hipLaunchKernelGGL((k_adj_curr<PM, CC>), dim3(nblk + (a->np + kBlock - 1) / kBlock), dim3(kBlock), 0, h->stream, h->g,
                       a->lI, a->B, a->A, h->kI, pI, a->lFI, nblk,
                       AdjSrc{a->lV, a->d_probes, a->np, a->freq, a->dT, ts, a->d_F});
    hipLaunchKernelGGL((k_adj_volt<PM, CC>), dim3(nblk), dim3(kBlock), 0, h->stream, h->g, a->lV, a->A, a->B, h->kV,
                       pV, a->lFV, a->box, hc, hv, a->gvi, a->gvv);
}

// one reverse step: the source of step ts, the transposed half steps
void adj_kernels(ems_adjoint* a, const float* hc, const float* hv, unsigned ts)
{
    ems_engine* h = a->h;
    const int pm = h->pmlV.n ? h->pml_mode : kNoPml;
    if (h->cmp) {
        if (pm == kPmlCompressed) adj_kernels_t<kPmlCompressed, true>(a, hc, hv, ts);
        else if (pm == kPmlPlain) adj_kernels_t<kPmlPlain, true>(a, hc, hv, ts);
        else adj_kernels_t<kNoPml, true>(a, hc, hv, ts);
    } else {
        if (pm == kPmlCompressed) adj_kernels_t<kPmlCompressed, false>(a, hc, hv, ts);
        else if (pm == kPmlPlain) adj_kernels_t<kPmlPlain, false>(a, hc, hv, ts);
        else adj_kernels_t<kNoPml, false>(a, hc, hv, ts);
    }
}

}  // namespace

extern "C" {

int ems_adj_create(ems_adjoint** out, ems_engine* h, unsigned nprobe, const unsigned* comp, const unsigned* pos,
                   const double* divisor, double freq, double dT, const unsigned box_lo[3], const unsigned box_hi[3],
                   unsigned checkpoint_every)
{
    if (!out || !h || !comp || !pos || !divisor || !box_lo || !box_hi) return fail(EMS_E_ARG, "null argument");
    *out = nullptr;
    if (!h->inited) return fail(EMS_E_STATE, "initialise the engine (ems_init) first");
    if (h->fused) return fail(EMS_E_ARG, "the adjoint runs the two-half-step form (ems_set_fused(h, 0))");
    if (!h->mur.empty() || !h->lor.empty() || !h->rlc.empty())
        return fail(EMS_E_ARG, "the adjoint supports UPML and sources only (no Mur, Lorentz, lumped RLC)");
    if (nprobe == 0 || !(dT > 0)) return fail(EMS_E_ARG, "no objective probes or bad timestep");
    if (checkpoint_every == 0) return fail(EMS_E_ARG, "checkpoint interval must be positive");
    AdjBox box{};
    box.x0 = box_lo[0];
    box.y0 = box_lo[1];
    box.z0 = box_lo[2];
    for (int n = 0; n < 3; ++n)
        if (box_hi[n] < box_lo[n] || box_hi[n] >= h->N[n]) return fail(EMS_E_ARG, "sensitivity box outside the mesh");
    box.nx = box_hi[0] - box_lo[0] + 1;
    box.ny = box_hi[1] - box_lo[1] + 1;
    box.nz = box_hi[2] - box_lo[2] + 1;
    box.n = (unsigned long long)box.nx * box.ny * box.nz;
    // the box must stay clear of the UPML (its coefficients are not the ones differentiated)
    for (int s = 0; s < h->pmlV.n; ++s) {
        const SlabTab& S = h->pmlV.tab[s];
        if ((int)box_lo[0] <= S.x1 && (int)box_hi[0] >= S.x0 && (int)box_lo[1] <= S.y1 && (int)box_hi[1] >= S.y0 &&
            (int)box_lo[2] <= S.z1 && (int)box_hi[2] >= S.z0)
            return fail(EMS_E_ARG, "the sensitivity box overlaps the UPML");
    }
    std::vector<AdjProbe> pr(nprobe);
    for (unsigned p = 0; p < nprobe; ++p) {
        const unsigned x = pos[p], y = pos[nprobe + p], z = pos[2 * nprobe + p];
        if (x >= h->N[0] || y >= h->N[1] || z >= h->N[2] || comp[p] > 2 || !(divisor[p] != 0.0))
            return fail(EMS_E_ARG, "objective probe outside the mesh or zero divisor");
        pr[p].lin = comp[p] * h->cs + h->lin(x, y, z);
        pr[p].div = divisor[p];
    }
    HIPCHK(hipSetDevice(h->device));
    ems_adjoint* a = new ems_adjoint();
    auto bail = [&](int r) {
        ems_adj_destroy(a);
        return r;
    };
    a->h = h;
    a->np = nprobe;
    a->freq = freq;
    a->dT = dT;
    a->box = box;
    a->K = checkpoint_every;
    int rc;
    const size_t c3 = 3 * h->cs;
    const size_t f3V = h->pmlV.n ? 3 * h->pmlV.npos : 1, f3I = h->pmlI.n ? 3 * h->pmlI.npos : 1;
    if ((rc = a->alloc(&a->d_probes, nprobe)) || (rc = a->alloc(&a->d_F, 2 * nprobe)) || (rc = a->alloc(&a->lV, c3)) ||
        (rc = a->alloc(&a->lI, c3)) || (rc = a->alloc(&a->A, c3)) || (rc = a->alloc(&a->B, c3)) ||
        (rc = a->alloc(&a->lFV, f3V)) || (rc = a->alloc(&a->lFI, f3I)) ||
        (rc = a->alloc(&a->gvi, 3 * box.n)) || (rc = a->alloc(&a->gvv, 3 * box.n)))
        return bail(rc);
    if (hipMemcpy(a->d_probes, pr.data(), nprobe * sizeof(AdjProbe), hipMemcpyHostToDevice) != hipSuccess)
        return bail(fail(EMS_E_HIP, "upload of the objective probes failed"));
    *out = a;
    return 0;
}

int ems_adj_forward(ems_adjoint* a, unsigned nsteps, double* J)
{
    TxRange tx("ems_adj_forward");
    if (!a || nsteps == 0) return fail(EMS_E_ARG, "null adjoint or no steps");
    ems_engine* h = a->h;
    HIPCHK(hipSetDevice(h->device));
    int rc;
    a->forward_done = false;     // until this run is: its records and saved states replace the last one's
    if ((rc = sync_probe_tables(h))) return rc;
    HIPCHK(hipStreamSynchronize(h->stream));
    HIPCHK(hipMemsetAsync(a->d_F, 0, 2 * a->np * sizeof(double), h->stream));
    a->n0 = h->numTS;
    a->nsteps = nsteps;
    const unsigned S = (nsteps + a->K - 1) / a->K;
    if (a->ck.size() < (size_t)S + 1) a->ck.resize(S + 1);
    if ((rc = adj_reserve(a, nsteps))) return rc;
    // with every step's record kept, the reverse pass needs no replay and so
    // no saved states on the way
    if (a->kept) adj_sample(a, 0, false);
    for (unsigned s = 0; s < S; ++s) {
        if (!a->kept && (rc = adj_save(a, a->ck[s]))) return rc;
        const unsigned len = std::min(a->K, nsteps - s * a->K);
        for (unsigned j = 0; j < len; ++j) {
            bool ahead = false;
            rc = launch_step(h, nullptr, false, ahead);
            ++h->numTS;
            if (rc) return rc;
            const unsigned n = s * a->K + j + 1;
            adj_sample(a, a->kept && n < nsteps ? (int)n : -1, true);
        }
    }
    if ((rc = adj_save(a, a->ck[S]))) return rc;
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(h->stream));
    a->F.assign(2 * a->np, 0.0);
    HIPCHK(hipMemcpy(a->F.data(), a->d_F, a->F.size() * sizeof(double), hipMemcpyDeviceToHost));
    double j = 0;
    for (unsigned p = 0; p < a->np; ++p) j += a->F[2 * p] * a->F[2 * p] + a->F[2 * p + 1] * a->F[2 * p + 1];
    if (J) *J = j;
    a->forward_done = true;
    return 0;
}

int ems_adj_backward(ems_adjoint* a, double* dJ_dvi, double* dJ_dvv)
{
    TxRange tx("ems_adj_backward");
    if (!a) return fail(EMS_E_ARG, "null adjoint");
    if (!a->forward_done) return fail(EMS_E_STATE, "run ems_adj_forward first");
    ems_engine* h = a->h;
    HIPCHK(hipSetDevice(h->device));
    const size_t c3 = 3 * h->cs * sizeof(float);
    HIPCHK(hipMemsetAsync(a->lV, 0, c3, h->stream));
    HIPCHK(hipMemsetAsync(a->lI, 0, c3, h->stream));
    HIPCHK(hipMemsetAsync(a->A, 0, c3, h->stream));
    HIPCHK(hipMemsetAsync(a->B, 0, c3, h->stream));
    if (h->pmlV.n) {
        HIPCHK(hipMemsetAsync(a->lFV, 0, 3 * h->pmlV.npos * sizeof(float), h->stream));
        HIPCHK(hipMemsetAsync(a->lFI, 0, 3 * h->pmlI.npos * sizeof(float), h->stream));
    }
    HIPCHK(hipMemsetAsync(a->gvi, 0, 3 * a->box.n * sizeof(double), h->stream));
    HIPCHK(hipMemsetAsync(a->gvv, 0, 3 * a->box.n * sizeof(double), h->stream));
    const unsigned S = (a->nsteps + a->K - 1) / a->K;
    int rc;
    for (int s = (int)S - 1; s >= 0; --s) {
        const unsigned len = std::min(a->K, a->nsteps - s * a->K);
        const size_t first = a->kept ? (size_t)s * a->K : 0;      // record of the segment's first step
        if (!a->kept) {
            // replay the segment, recording the inputs of each voltage update
            if ((rc = adj_restore(a, a->ck[s]))) return rc;
            for (unsigned j = 0; j < len; ++j) {
                adj_sample(a, (int)j, false);
                bool ahead = false;
                rc = launch_step(h, nullptr, false, ahead);
                ++h->numTS;
                if (rc) return rc;
            }
        }
        // reverse steps of the segment
        for (int j = (int)len - 1; j >= 0; --j) {
            const size_t at = (first + (size_t)j) * 3 * a->box.n;
            adj_kernels(a, a->hc + at, a->hv + at, a->n0 + (unsigned)s * a->K + (unsigned)j + 1);
        }
    }
    HIPCHK(hipGetLastError());
    // leave the engine at the end of the forward run
    if ((rc = adj_restore(a, a->ck[S]))) return rc;
    if (dJ_dvi) HIPCHK(hipMemcpy(dJ_dvi, a->gvi, 3 * a->box.n * sizeof(double), hipMemcpyDeviceToHost));
    if (dJ_dvv) HIPCHK(hipMemcpy(dJ_dvv, a->gvv, 3 * a->box.n * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

int ems_adj_get_records(const ems_adjoint* a, int* kept, unsigned long long* steps)
{
    if (!a) return fail(EMS_E_ARG, "null adjoint");
    if (kept) *kept = a->kept ? 1 : 0;
    if (steps) *steps = a->rec_steps;
    return 0;
}

void ems_adj_destroy(ems_adjoint* a)
{
    if (!a) return;
    if (a->h) {
        hipSetDevice(a->h->device);
        if (a->h->stream) hipStreamSynchronize(a->h->stream);
    }
    for (void* p : a->allocs) hipFree(p);
    if (a->hc) hipFree(a->hc);
    if (a->hv) hipFree(a->hv);
    delete a;
}

}  // extern "C"
