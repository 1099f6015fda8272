// Per-cell device code of the compact layout shared by its step kernels:
// storage conversions, the pull with its boundary handling, the FP32
// arithmetic of the shifted storage, and the host code that fills the
// kernels' argument structures.  Everything has internal linkage.
#pragma once

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>

#include "mrb_internal.h"

namespace mrb {
namespace {

struct CompactArgs {
    int nx, ny, nz;
    int per[3];
    int64_t N;   // cells
    int64_t cs;  // component stride of the population arrays (2N)
    int bc[6];
    uint32_t bcpack;  // bc[face] in bits 4*face .. 4*face+3
    int fast_ok;      // byte offsets of a lattice's cells fit 32 bits
};

// Source coordinates of the pull for one direction component c in
// {-1,0,1} along a dimension of extent n.  Returns false when the source
// lies beyond a non-periodic face (a physical-boundary ghost).
__device__ __forceinline__ void wrap3(int x, int n, int periodic, int s[3], bool ghost[3])
{
    // index c+1: source x - c
    s[0] = x + 1;  // c = -1
    s[1] = x;      // c = 0
    s[2] = x - 1;  // c = +1
    ghost[0] = ghost[1] = ghost[2] = false;
    if (s[0] >= n) {
        if (periodic)
            s[0] -= n;
        else
            ghost[0] = true;
    }
    if (s[2] < 0) {
        if (periodic)
            s[2] += n;
        else
            ghost[2] = true;
    }
}

// Rest-state populations subtracted by the shifted storages (stored value =
// population - shift); one value per speed class |c_q|^2 = 0..3, so the
// eight values sit in scalar registers; unused for FP64 storage.
struct ShiftTab {
    double fk[4], gk[4];
    __device__ __forceinline__ double f(int q) const { return fk[csq(q)]; }
    __device__ __forceinline__ double g(int q) const { return gk[csq(q)]; }
};

// Rest state of the shifted FP32 storage, for its FP32-arithmetic collide
// (k_collide_f32): the product-form factors and the Grad coefficients of
// the subtracted equilibrium f_eq(rho0, 0, T0), g_eq(rho0, 0, T0), and the
// raw moments of those shifts; FP64.
struct DevRest {
    double A0[3];   // rho0 phi0(c), c = -1, 0, 1 (the shift's x factor)
    double B0[3];   // phi0(c) (its y and z factors)
    double E0;      // 2 rho0 E of the rest state
    double t0[2];   // (c^2 - theta0) a2_aa of the rest state, c^2 = 0, 1
    double mo[14];  // moments of the shifts, in MomentsR order
};

// Element stride between neighbouring cells of one component: every
// storage keeps f_q and g_q of a cell side by side
// (pop[(q*N + cell)*2 + lattice]) so that one load or store moves both.
template <class T>
constexpr int kCellStride = 2;
template <class T>
constexpr bool kIsHalf = std::is_same<T, _Float16>::value;

// store of a cell's f_q and g_q
template <class T>
__device__ __forceinline__ void store_pair(T *__restrict__ fo, T *__restrict__ go, int64_t e, T fv, T gv)
{
    if constexpr (kIsHalf<T>) {
        (void)go;
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        h2 v;
        v.x = fv;
        v.y = gv;
        *reinterpret_cast<h2 *>(fo + e) = v;
    } else if constexpr (std::is_same<T, double>::value) {
        // non-temporal: the next step reads the buffer back from HBM
        // (measured at 256^3: z-sweep 3.039 -> 3.024 ms FP64, 2.34 -> 2.30 ms
        // shifted FP32)
        (void)go;
        typedef double d2 __attribute__((ext_vector_type(2)));
        d2 v;
        v.x = fv;
        v.y = gv;
        __builtin_nontemporal_store(v, reinterpret_cast<d2 *>(fo + e));
    } else {
        (void)go;
        typedef float f2 __attribute__((ext_vector_type(2)));
        f2 v;
        v.x = fv;
        v.y = gv;
        __builtin_nontemporal_store(v, reinterpret_cast<f2 *>(fo + e));
    }
}

// load of a cell's f_q and g_q: one 16-byte (FP64), 8-byte (FP32) or
// 4-byte (FP16) access; NT: the values are not read again before they are
// overwritten, so they need not stay in the caches
template <bool NT, class T>
__device__ __forceinline__ void load_stored_pair(const T *__restrict__ p, T &fv, T &gv)
{
    if constexpr (kIsHalf<T>) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const uint32_t *u = reinterpret_cast<const uint32_t *>(p);
        uint32_t w;
        if constexpr (NT)
            w = __builtin_nontemporal_load(u);
        else
            w = *u;
        const h2 v = __builtin_bit_cast(h2, w);
        fv = v.x;
        gv = v.y;
    } else {
        typedef T t2 __attribute__((ext_vector_type(2)));
        const t2 *u = reinterpret_cast<const t2 *>(p);
        t2 v;
        if constexpr (NT)
            v = __builtin_nontemporal_load(u);
        else
            v = *u;
        fv = v.x;
        gv = v.y;
    }
}

// FP16 storage: scale exponents and box maxima of the read (cur) and the
// written (next) buffers, per (scale box, lattice); unused by the other
// storages
struct Half16 {
    const int *__restrict__ e_cur;
    int *__restrict__ e_next;
    const uint32_t *__restrict__ amax_cur;
    uint32_t *__restrict__ amax_next;
    uint32_t *__restrict__ ovf;
    // the largest |population - shift| the boundary faces bring in (inlet
    // and pressure-face equilibria), per lattice: a lower bound for the box
    // maxima that set the next scales, so that a box at rest next to an
    // inlet keeps room for the inflow
    float floor_f, floor_g;
};

// Largest |population - shift| that scale box b's written cells can be
// pulled from: the maxima of boxes b-1, b and b+1 in the read buffer (a pull
// reaches one plane into each neighbouring box; the neighbours wrap on a
// periodic z axis), no smaller than the boundary floor.  A box exactly at
// the shift state (maximum 0) next to a disturbed one thereby takes the
// disturbed box's scale instead of the largest exponent.
__device__ __forceinline__ float f16_pull_max(const uint32_t *__restrict__ amax, int b, int lattice, int nz,
                                              int periodic_z, float floor)
{
    const int nb = (nz + kScaleSlab - 1) / kScaleSlab;
    float m = fmaxf(__uint_as_float(amax[2 * b + lattice]), floor);
    int bm = b - 1, bp = b + 1;
    if (periodic_z) {
        bm = bm < 0 ? nb - 1 : bm;
        bp = bp >= nb ? 0 : bp;
    }
    if (bm >= 0) m = fmaxf(m, __uint_as_float(amax[2 * bm + lattice]));
    if (bp < nb) m = fmaxf(m, __uint_as_float(amax[2 * bp + lattice]));
    return m;
}

// FP16 value of (v - shift) * scale, scale a power of two: the difference
// is taken in the type of v, then rounded to FP32 and clamped there to the
// values whose FP16 counterpart is finite (lim = 65504 / scale, exact), then
// scaled (exact) and rounded; amax tracks |v - shift|
template <class V>
__device__ __forceinline__ _Float16 to_half(V v, V shift, float scale, float lim, float &amax)
{
    const float d = float(v - shift);
    amax = fmaxf(amax, fabsf(d));
    return _Float16(__builtin_fmaf(__builtin_amdgcn_fmed3f(d, -lim, lim), scale, 0.0f));
}

// storage <-> FP64 working value (FP64 and shifted FP32 storage)
template <class T>
__device__ __forceinline__ double widen(T v, double shift)
{
    if constexpr (std::is_same<T, double>::value) {
        (void)shift;
        return v;
    } else {
        return double(v) + shift;
    }
}
template <class T>
__device__ __forceinline__ T narrow(double v, double shift)
{
    if constexpr (std::is_same<T, double>::value) {
        (void)shift;
        return v;
    } else {
        return T(v - shift);
    }
}

// Per dimension, for the three lattice-velocity components c = -1, 0, +1
// (index c + 1): t = the coordinate the pull reads, x - c wrapped on a
// periodic axis and, beyond a non-periodic face, the boundary cell next to
// the ghost (the cell an outflow ghost copies); g = the source is a ghost.
// the directions q with c_q[d] == c, as a bit set
constexpr uint32_t qset(int d, int c)
{
    uint32_t m = 0;
    for (int q = 0; q < NQ; ++q)
        if (ev(q, d) == c) m |= 1u << q;
    return m;
}
constexpr uint32_t kAllQ = (1u << NQ) - 1u;

__device__ __forceinline__ void targets3(int x, int n, int periodic, int t[3], bool g[3])
{
    const int p = x + 1, m = x - 1;
    const bool hi = p >= n, lo = m < 0;
    g[0] = hi && !periodic;
    g[1] = false;
    g[2] = lo && !periodic;
    t[0] = hi ? (periodic ? p - n : n - 1) : p;
    t[1] = x;
    t[2] = lo ? (periodic ? m + n : 0) : m;
}

// the directions with c_q[d] == c, in order
constexpr int qwith(int d, int c, int k)
{
    for (int q = 0; q < NQ; ++q)
        if (ev(q, d) == c && k-- == 0) return q;
    return -1;
}

// Compile-time boundary features of a level's pull (template argument BCX):
// a Channel or Parabolic inlet profile, PRESSURE faces
constexpr int kBcxProfile = 1;
constexpr int kBcxPressure = 2;
// the profile inlet's only VELOCITY face is x-lo, as in the channel and duct
// workloads and the 660x123x4 cylinder deck: the lookups of the other faces,
// merged into one pull, take the FP64 passes from 150 and 200 registers to 228
// and 239.  (The 246x576x4 deck's inlet at y-lo takes them: 141 us per step.)
constexpr int kBcxProfileX = 4;

// pressure_bc_f (BC.H:222-271) for the fluid cell (x, y, z) next to a
// PRESSURE face of axis pd: the ghosts of the directions in Pm take
// f_eq(rho_bc, u, R T) with u along pd from the populations the cell
// receives.  The reference reads them as data(x + c_qq, qqbar): for the
// tangential and outgoing directions those are the pulled values (a
// periodic image, or a NOSLIP ghost whose value is the cell's own
// population), except from a solid cell, which holds its stored value (0
// in the initial state, the -1 of the stream afterwards; FP16 storage keeps
// 0 there, so -1 is used)
template <class T>
__device__ __forceinline__ void pressure_ghosts(
    const T *__restrict__ f, const CompactArgs &A, const BCDev &bc, const ShiftTab &sh, const int tx[3],
    const int ty[3], const int tz[3], int x, int y, int z, uint32_t mask, uint32_t Pm, double fv[NQ],
    double gv[NQ])
{
    const int pd = bc.pdir;
    const int xc = pd == 0 ? x : (pd == 1 ? y : z);
    const int ndir = xc == 0 ? 1 : -1;
    double rho_out = 0.0, rho_tan = 0.0;
    static_for<NQ>([&](auto qc) {
        constexpr int qq = decltype(qc)::value;
        constexpr int p = kBounce[qq];
        constexpr int cx = ev(p, 0), cy = ev(p, 1), cz = ev(p, 2);
        const int cin = pd == 0 ? cx : (pd == 1 ? cy : cz);
        if (cin == -ndir || cin == 0) {
            double v = fv[p];
            if (!((mask >> p) & 1u)) {
                if constexpr (kIsHalf<T>) {
                    v = -1.0;
                } else {
                    const int64_t src =
                        (int64_t(tz[cz + 1]) * A.ny + ty[cy + 1]) * A.nx + tx[cx + 1];
                    v = widen(f[int64_t(p) * A.cs + src * kCellStride<T>], sh.f(p));
                }
            }
            if (cin == -ndir)
                rho_out += 2.0 * v;
            else
                rho_tan += 1.0 * v;
        }
    });
    const double un = ndir * (1.0 - (rho_out + rho_tan) / bc.prho);
    const double vel[3] = {pd == 0 ? un : 0.0, pd == 1 ? un : 0.0, pd == 2 ? un : 0.0};
    static_for<NQ>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if ((Pm >> q) & 1u) {
            fv[q] = set_equilibrium_value(bc.prho, vel, bc.prt, q);
            gv[q] = bc.pgval[q];
        }
    });
}

// The boundary handling of the 27 sources as bit sets over q, per cell.
// BCFill applies the faces a ghost lies beyond in the order x, y, z, the
// last one winning (BC.H:365-372); an OUTFLOW face copies the ghost one
// step inward, whose own value the remaining faces set (the ghosts are
// filled in order of their distance beyond the domain).  So, scanning
// z, y, x: G = sources beyond a non-periodic face; Tm = those whose value
// a non-OUTFLOW face fixes (the first such face in the scan), with V, Pm
// the VELOCITY and PRESSURE ones; O = the rest of G, beyond OUTFLOW
// faces only, which read the source clamped into the domain.  A source
// is read directly unless it is a solid cell or Tm holds it with a wall.
struct SourceSets {
    uint32_t G, Tm, V, Pm;
    // the sources not read directly; mask: the cell's stream mask
    __device__ __forceinline__ uint32_t nondirect(uint32_t mask) const
    {
        const uint32_t O = G & ~Tm;
        return (G & ~(V | O)) | (~G & ~mask & kAllQ);
    }
};
template <int BCX>
__device__ __forceinline__ SourceSets source_sets(const CompactArgs &A, const bool gx[3], const bool gy[3],
                                                  const bool gz[3])
{
    uint32_t G = 0, Tm = 0, V = 0, Pm = 0;
    static_for<3>([&](auto dc) {
        constexpr int d = 2 - decltype(dc)::value;
        const bool *gd = d == 0 ? gx : (d == 1 ? gy : gz);
        const uint32_t Gd = (gd[2] ? qset(d, 1) : 0u) | (gd[0] ? qset(d, -1) : 0u);
        const uint32_t Ud = Gd & ~Tm;
        G |= Gd;
        const uint32_t tl = (A.bcpack >> (4 * d)) & 15u, th = (A.bcpack >> (4 * (d + 3))) & 15u;
        const uint32_t lo = Ud & qset(d, 1), hi = Ud & qset(d, -1);
        Tm |= (tl != MRB_BC_OUTFLOW ? lo : 0u) | (th != MRB_BC_OUTFLOW ? hi : 0u);
        V |= (tl == MRB_BC_VELOCITY ? lo : 0u) | (th == MRB_BC_VELOCITY ? hi : 0u);
        if constexpr ((BCX & kBcxPressure) != 0)
            Pm |= (tl == MRB_BC_PRESSURE ? lo : 0u) | (th == MRB_BC_PRESSURE ? hi : 0u);
    });
    return SourceSets{G, Tm, V, Pm};
}

// Pull of one cell, without branches so that all 54 loads are in flight
// together.  For a pull source beyond a physical face the reference's
// BCFill value is resolved: the face applied is the last non-periodic face
// in BCFill's loop order (BC.H:365-372, z over y over x); NOSLIP and SLIP
// read the cell's own pre-stream populations, OUTFLOW the boundary cell
// next to the ghost (at a corner of two non-periodic faces, clamped in
// both), VELOCITY a constant.
// W = the working type of the pulled values (double); BCX: the level's
// boundary features (kBcxProfile: Channel or Parabolic inlet profile, ghost
// values from the face tables; kBcxPressure: PRESSURE faces)
// DEV (shifted FP32 storage only): return the stored deviations f - shift
// themselves (boundary constants less the shift) instead of populations.
// The pull in two phases: pull_raw issues the loads of the stored values
// (rf, rg) and returns which sources take a boundary constant (cmask), are
// read directly (dmask), were moved inward across a z OUTFLOW face (zmove)
// or lie beyond a PRESSURE face (Pm); pull_finish turns them into
// populations.  A caller with other work to do (the z-sweep) places that
// work between the two, so that the loads stay in flight meanwhile.
struct PullBits {
    uint32_t cmask, dmask, zmove, Pm;
};

template <int BCX, class T, bool UNIFORM_LOADS = false, bool NT = false>
__device__ __forceinline__ PullBits pull_raw(
    const T *__restrict__ f, const CompactArgs &A, int x, int y, int z, int64_t cell, uint32_t mask, T rf[NQ],
    T rg[NQ])
{
    int tx[3], ty[3], tz[3];
    bool gx[3], gy[3], gz[3];
    targets3(x, A.nx, A.per[0], tx, gx);
    targets3(y, A.ny, A.per[1], ty, gy);
    targets3(z, A.nz, A.per[2], tz, gz);
    const uint32_t c32 = uint32_t(cell);
    uint32_t cmask = 0, dmask = 0, zmove = 0;
    const SourceSets S = source_sets<BCX>(A, gx, gy, gz);
    const uint32_t G = S.G, V = S.V, Pm = S.Pm;
    const uint32_t nondirect = S.nondirect(mask);
    (void)G;
    // one (f_q, g_q) pair from element e of the f buffer (g == f + 1)
    auto load_pair = [&](int q, int64_t e) { load_stored_pair<NT>(f + e, rf[q], rg[q]); };
    // the element of direction q's source on the general path: the pull's
    // source, its bounce-back, a reflection or a cell moved inward
    auto general_e = [&](auto qc) -> int64_t {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
        constexpr int qb = kBounce[q];
        const bool hx = gx[cx + 1], hy = gy[cy + 1], hz = gz[cz + 1];
        const bool ghost = hx || hy || hz;
        const uint32_t src = (uint32_t(tz[cz + 1]) * uint32_t(A.ny) + uint32_t(ty[cy + 1])) * uint32_t(A.nx) +
                             uint32_t(tx[cx + 1]);
        // the face that fixes a ghost source's value (scan z, y, x past
        // OUTFLOW faces, as above) and the cell its wall fill reads: the cell
        // itself moved one step inward across each OUTFLOW face passed
        const uint32_t tfz = (A.bcpack >> (4 * (cz > 0 ? 2 : 5))) & 15u;
        const uint32_t tfy = (A.bcpack >> (4 * (cy > 0 ? 1 : 4))) & 15u;
        const uint32_t tfx = (A.bcpack >> (4 * (cx > 0 ? 0 : 3))) & 15u;
        const bool pz = hz && tfz == MRB_BC_OUTFLOW;
        const bool py = hy && tfy == MRB_BC_OUTFLOW && (pz || !hz);
        const bool px = hx && tfx == MRB_BC_OUTFLOW && (py || !hy) && (pz || !hz);
        const uint32_t t = (hz && !pz) ? tfz : (hy && !py) ? tfy : (hx && !px) ? tfx : uint32_t(MRB_BC_OUTFLOW);
        const int32_t roff = (pz ? cz * A.nx * A.ny : 0) + (py ? cy * A.nx : 0) + (px ? cx : 0);
        zmove |= uint32_t(pz) << q;
        const bool direct = ghost ? t == MRB_BC_OUTFLOW : ((mask >> q) & 1u) != 0;
        int comp = direct ? q : qb;
        comp = (ghost && t == MRB_BC_SLIPX) ? reflect(q, 0) : comp;
        comp = (ghost && t == MRB_BC_SLIPY) ? reflect(q, 1) : comp;
        comp = (ghost && t == MRB_BC_SLIPZ) ? reflect(q, 2) : comp;
        dmask |= uint32_t(direct) << q;
        cmask |= uint32_t(ghost && t == MRB_BC_VELOCITY) << q;
        return int64_t(comp) * A.cs + int64_t(direct ? src : uint32_t(int32_t(c32) + roff)) * kCellStride<T>;
    };
    const bool all_direct = __all(nondirect == 0u);
    if constexpr (UNIFORM_LOADS) {
        // the 27 source elements on the direct path or the general one (no
        // memory access on either), then the loads in one fixed sequence:
        // the number of loads in flight is then the same on every path
        int64_t e[NQ];
        if (all_direct) {
            const uint32_t nxy = uint32_t(A.nx) * uint32_t(A.ny);
            uint32_t xi[3], yi[3], zi[3];
            for (int k = 0; k < 3; ++k) {
                xi[k] = uint32_t(tx[k]);
                yi[k] = uint32_t(ty[k]) * uint32_t(A.nx);
                zi[k] = uint32_t(tz[k]) * nxy;
            }
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
                e[q] = int64_t(q) * A.cs + int64_t(zi[cz + 1] + yi[cy + 1] + xi[cx + 1]) * kCellStride<T>;
            });
            cmask = V;
            dmask = kAllQ;
        } else {
            static_for<NQ>([&](auto qc) { e[decltype(qc)::value] = general_e(qc); });
        }
        static_for<NQ>([&](auto qc) { load_pair(decltype(qc)::value, e[decltype(qc)::value]); });
    } else if (A.fast_ok && all_direct) {
        // every source of every cell of the wave is read directly: one
        // wave-uniform base per direction and a 32-bit byte offset per lane
        constexpr uint32_t bytes = kCellStride<T> * sizeof(T);
        const uint32_t nxb = uint32_t(A.nx) * bytes, nxyb = nxb * uint32_t(A.ny);
        uint32_t xo[3], yo[3], zo[3];
        for (int k = 0; k < 3; ++k) {
            xo[k] = uint32_t(tx[k]) * bytes;
            yo[k] = uint32_t(ty[k]) * nxb;
            zo[k] = uint32_t(tz[k]) * nxyb;
        }
        static_for<NQ>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
            const uint32_t off = zo[cz + 1] + yo[cy + 1] + xo[cx + 1];
            const char *bf = reinterpret_cast<const char *>(f) + int64_t(q) * A.cs * int64_t(sizeof(T));
            load_stored_pair<NT>(reinterpret_cast<const T *>(bf + off), rf[q], rg[q]);
        });
        cmask = V;
        dmask = kAllQ;
    } else {
        static_for<NQ>([&](auto qc) { load_pair(decltype(qc)::value, general_e(qc)); });
    }
    return PullBits{cmask, dmask, zmove, Pm};
}

// The loads of the pull before the cell's stream mask is known: every source
// read as if it were fluid (clamped into the domain beyond a non-periodic
// face), in one fixed sequence without a branch.  pull_settle, given the
// mask, keeps them where the source is read directly and loads the others
// (walls, solid sources) again, lane by lane.  Repeating the whole pull of a wave
// with one such source took more than the mask's latency had cost: 96x64x48
// cells between six walls, FP64, 101 us per step against 86 (88 on row blocks,
// whose pull waits for the mask); 160x120x100 with a pressure outlet, whose
// ghosts need no second load, 510 against 404.
template <class T, bool NT>
__device__ __forceinline__ void pull_ahead(const T *__restrict__ f, const CompactArgs &A, int x, int y, int z,
                                           T rf[NQ], T rg[NQ])
{
    int tx[3], ty[3], tz[3];
    bool gx[3], gy[3], gz[3];
    targets3(x, A.nx, A.per[0], tx, gx);
    targets3(y, A.ny, A.per[1], ty, gy);
    targets3(z, A.nz, A.per[2], tz, gz);
    // z is the same for the whole wave: a scalar base per direction and a
    // 32-bit byte offset within the plane per lane
    constexpr uint32_t bytes = kCellStride<T> * sizeof(T);
    const uint32_t nxb = uint32_t(A.nx) * bytes;
    uint32_t xo[3], yo[3];
    const char *zb[3];
    for (int k = 0; k < 3; ++k) {
        xo[k] = uint32_t(tx[k]) * bytes;
        yo[k] = uint32_t(ty[k]) * nxb;
        zb[k] = reinterpret_cast<const char *>(f) + int64_t(tz[k]) * A.ny * int64_t(nxb);
    }
    static_for<NQ>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
        const char *b = zb[cz + 1] + int64_t(q) * A.cs * int64_t(sizeof(T));
        load_stored_pair<NT>(reinterpret_cast<const T *>(b + (yo[cy + 1] + xo[cx + 1])), rf[q], rg[q]);
    });
}
// The element that direction q's source is read from when it is a wall's ghost or
// a solid cell, as pull_raw's general path resolves it (kept apart from it: the
// z-sweep on FP32 storage lost 10 % when it took its elements from here).  pz:
// the cell read was moved inward across a z OUTFLOW face.
template <int q, class T>
__device__ __forceinline__ int64_t wall_e(const CompactArgs &A, const bool gx[3], const bool gy[3], const bool gz[3],
                                          int64_t cell, bool &pz)
{
    constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
    const bool hx = gx[cx + 1], hy = gy[cy + 1], hz = gz[cz + 1];
    const uint32_t tfz = (A.bcpack >> (4 * (cz > 0 ? 2 : 5))) & 15u;
    const uint32_t tfy = (A.bcpack >> (4 * (cy > 0 ? 1 : 4))) & 15u;
    const uint32_t tfx = (A.bcpack >> (4 * (cx > 0 ? 0 : 3))) & 15u;
    pz = hz && tfz == MRB_BC_OUTFLOW;
    const bool py = hy && tfy == MRB_BC_OUTFLOW && (pz || !hz);
    const bool px = hx && tfx == MRB_BC_OUTFLOW && (py || !hy) && (pz || !hz);
    const uint32_t t = (hz && !pz) ? tfz : (hy && !py) ? tfy : (hx && !px) ? tfx : uint32_t(MRB_BC_OUTFLOW);
    const int32_t roff = (pz ? cz * A.nx * A.ny : 0) + (py ? cy * A.nx : 0) + (px ? cx : 0);
    int comp = kBounce[q];
    comp = t == MRB_BC_SLIPX ? reflect(q, 0) : comp;
    comp = t == MRB_BC_SLIPY ? reflect(q, 1) : comp;
    comp = t == MRB_BC_SLIPZ ? reflect(q, 2) : comp;
    return int64_t(comp) * A.cs + int64_t(uint32_t(int32_t(uint32_t(cell)) + roff)) * kCellStride<T>;
}

template <int BCX, class T, bool NT>
__device__ __forceinline__ PullBits pull_settle(const T *__restrict__ f, const CompactArgs &A, int x, int y, int z,
                                                int64_t cell, uint32_t mask, T rf[NQ], T rg[NQ])
{
    // away from non-periodic faces and solid cells nothing is left to do
    const bool edge = (!A.per[0] && (x == 0 || x == A.nx - 1)) || (!A.per[1] && (y == 0 || y == A.ny - 1)) ||
                      (!A.per[2] && (z == 0 || z == A.nz - 1));
    PullBits pb{0u, kAllQ, 0u, 0u};
    if (__any(edge || mask != kAllQ)) {
        int tx[3], ty[3], tz[3];
        bool gx[3], gy[3], gz[3];
        targets3(x, A.nx, A.per[0], tx, gx);
        targets3(y, A.ny, A.per[1], ty, gy);
        targets3(z, A.nz, A.per[2], tz, gz);
        const SourceSets S = source_sets<BCX>(A, gx, gy, gz);
        pb.cmask = S.V;
        pb.Pm = S.Pm;
        // (a PRESSURE ghost's value replaces what was loaded)
        const uint32_t nd = S.nondirect(mask) & ~S.Pm;
        pb.dmask = kAllQ & ~nd;
        if (__any(nd != 0u)) {
            // An FP32 pair is kept as one word meanwhile: as two values the
            // compiler may copy each pair behind its load, which then waits
            // for it (pass 2 of a y-lo profile inlet, 246x576x4: 98 us per step
            // against 88); of an FP16 pair the word costs more scratch
            struct Pair {
                T f, g;
            };
            using Bits = std::conditional_t<std::is_same<T, float>::value, uint64_t, Pair>;
            constexpr bool kWord = std::is_same<T, float>::value;
            Bits word[NQ];
            if constexpr (kWord)
                for (int q = 0; q < NQ; ++q) word[q] = __builtin_bit_cast(Bits, Pair{rf[q], rg[q]});
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if ((nd >> q) & 1u) {
                    bool pz;
                    Pair v;
                    load_stored_pair<NT>(f + wall_e<q, T>(A, gx, gy, gz, cell, pz), v.f, v.g);
                    pb.zmove |= uint32_t(pz) << q;
                    if constexpr (kWord) {
                        word[q] = __builtin_bit_cast(Bits, v);
                    } else {
                        rf[q] = v.f;
                        rg[q] = v.g;
                    }
                }
            });
            if constexpr (kWord)
                for (int q = 0; q < NQ; ++q) {
                    asm volatile("" : "+v"(word[q]));
                    const Pair v = __builtin_bit_cast(Pair, word[q]);
                    rf[q] = v.f;
                    rg[q] = v.g;
                }
        }
    }
    return pb;
}

template <int BCX, class T, class W, bool DEV = false>
__device__ __forceinline__ void pull_finish(
    const T *__restrict__ f, const CompactArgs &A, const BCDev &bc, const ShiftTab &sh, const Half16 &h16,
    int x, int y, int z, uint32_t mask, const PullBits &pb, const T rf[NQ], const T rg[NQ], W fv[NQ], W gv[NQ])
{
    static_assert(!DEV || (std::is_same<T, float>::value && (BCX & kBcxPressure) == 0),
                  "deviation pull: shifted FP32 storage without PRESSURE faces");
    int tx[3], ty[3], tz[3];
    bool gx[3], gy[3], gz[3];
    targets3(x, A.nx, A.per[0], tx, gx);
    targets3(y, A.ny, A.per[1], ty, gy);
    targets3(z, A.nz, A.per[2], tz, gz);
    const uint32_t cmask = pb.cmask, dmask = pb.dmask, zmove = pb.zmove, Pm = pb.Pm;
    (void)zmove;
    (void)tx;
    (void)ty;
    if constexpr (kIsHalf<T>) {
        // inverse scales of the source planes z - c_z (index c_z + 1); a
        // source that is not the pull's (bounce-back, wall ghosts) is the
        // cell itself, in plane z (index 1).  Wave-uniform values.
        float invf[3], invg[3];
        for (int k = 0; k < 3; ++k) {
            const int b = tz[k] / kScaleSlab;
            invf[k] = ldexpf(1.0f, -h16.e_cur[2 * b]);
            invg[k] = ldexpf(1.0f, -h16.e_cur[2 * b + 1]);
        }
        // unscaling in FP32 is exact (a power of two on an FP16 value)
        auto unscale = [&](T h, float scale, double shift) -> W {
            if constexpr (std::is_same<W, float>::value)
                return __builtin_fmaf(float(h), scale, float(shift));
            else
                return double(__builtin_fmaf(float(h), scale, 0.0f)) + shift;
        };
        if (__all(dmask == kAllQ)) {
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                constexpr int k = ev(q, 2) + 1;
                fv[q] = unscale(rf[q], invf[k], sh.f(q));
                gv[q] = unscale(rg[q], invg[k], sh.g(q));
            });
        } else {
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                constexpr int k = ev(q, 2) + 1;
                const bool direct = (dmask >> q) & 1u;
                // a wall fill read moved inward across a z OUTFLOW face lies in
                // plane z + c_z (index 1 - c_z)
                constexpr int km = 1 - ev(q, 2);
                const bool moved = (zmove >> q) & 1u;
                fv[q] = unscale(rf[q], direct ? invf[k] : (moved ? invf[km] : invf[1]), sh.f(q));
                gv[q] = unscale(rg[q], direct ? invg[k] : (moved ? invg[km] : invg[1]), sh.g(q));
            });
        }
    } else {
        (void)dmask;
        static_for<NQ>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (DEV) {
                fv[q] = W(rf[q]);
                gv[q] = W(rg[q]);
            } else {
                fv[q] = widen(rf[q], sh.f(q));
                gv[q] = widen(rg[q], sh.g(q));
            }
        });
    }
    // The boundary constants, behind one branch that only the waves next to
    // an inlet face enter: selected direction by direction in every wave they
    // cost 6 instructions per direction and pass, a seventh of the FP64 step's
    if (__any(cmask != 0u)) {
        if constexpr ((BCX & kBcxProfile) != 0) {
            // Table lookups of a profile inlet, face by face, the loads of a
            // face's 9 directions in flight together (the entry of the ghost
            // cell x - c_q: every lane's index lies in the table).  Looked up
            // one after the other, each under its lanes' own branch, the
            // waves next to the inlet (two in five on 160-cell rows) waited
            // for nine of them in turn.  A ghost beyond several faces belongs
            // to the last of x, y, z (BCFill's loop order); mrb_set_bc refuses
            // an OUTFLOW face on an axis after the inlet's, which would copy
            // another ghost's value here.
            static_for<(BCX & kBcxProfileX) != 0 ? 1 : 6>([&](auto fc) {
                constexpr int face = decltype(fc)::value, d = face % 3, c = face < 3 ? 1 : -1;
                constexpr int d1 = d == 0 ? 1 : 0, d2 = d == 2 ? 1 : 2;
                if (bc.tab[face]) {
                    uint32_t own = cmask & qset(d, c);
                    if (d < 2) own &= ~((gz[2] ? qset(2, 1) : 0u) | (gz[0] ? qset(2, -1) : 0u));
                    if (d < 1) own &= ~((gy[2] ? qset(1, 1) : 0u) | (gy[0] ? qset(1, -1) : 0u));
                    if (__any(own != 0u)) {
                        const int t1 = d1 == 0 ? x : y, t2 = d2 == 1 ? y : z;
                        const int w = bc.tabw[face], e0 = (t1 + 1) * w + t2 + 1;
                        double tf[9], tg[9];
                        static_for<9>([&](auto kc) {
                            constexpr int k = decltype(kc)::value, q = qwith(d, c, k);
                            const double *t = bc.tab[face] + int64_t(e0 - (ev(q, d1) * w + ev(q, d2))) * (2 * NQ);
                            tf[k] = t[q];
                            tg[k] = t[NQ + q];
                        });
                        static_for<9>([&](auto kc) {
                            constexpr int k = decltype(kc)::value, q = qwith(d, c, k);
                            const bool use_const = (own >> q) & 1u;
                            fv[q] = use_const ? (DEV ? W(tf[k] - sh.f(q)) : W(tf[k])) : fv[q];
                            gv[q] = use_const ? (DEV ? W(tg[k] - sh.g(q)) : W(tg[k])) : gv[q];
                        });
                    }
                }
            });
        } else {
            static_for<NQ>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                const bool use_const = (cmask >> q) & 1u;
                const double cf = bc.fval[q], cg = bc.gval[q];
                fv[q] = use_const ? (DEV ? W(cf - sh.f(q)) : W(cf)) : fv[q];
                gv[q] = use_const ? (DEV ? W(cg - sh.g(q)) : W(cg)) : gv[q];
            });
        }
    }
    if constexpr ((BCX & kBcxPressure) != 0) {
        // (a cell with a PRESSURE ghost source never takes the fast path)
        if (Pm) pressure_ghosts(f, A, bc, sh, tx, ty, tz, x, y, z, mask, Pm, fv, gv);
    } else {
        (void)Pm;
    }
}

template <int BCX, class T, class W, bool DEV = false, bool NT = false>
__device__ __forceinline__ void pull_cell(
    const T *__restrict__ f, const T *__restrict__ g, const CompactArgs &A, const BCDev &bc,
    const ShiftTab &sh, const Half16 &h16, int x, int y, int z, int64_t cell, uint32_t mask, W fv[NQ],
    W gv[NQ])
{
    (void)g;  // g == f + 1 (f_q and g_q of a cell side by side)
    T rf[NQ], rg[NQ];
    const PullBits pb = pull_raw<BCX, T, false, NT>(f, A, x, y, z, cell, mask, rf, rg);
    pull_finish<BCX, T, W, DEV>(f, A, bc, sh, h16, x, y, z, mask, pb, rf, rg, fv, gv);
}

// The six neighbours' Q_corr of a cell, loaded unconditionally with the
// pull (indices clamped into the domain: a value past a face is loaded but
// not used), so that the gradient does not wait on loads issued after the
// moments.
struct QNbr {
    double xp, xm, yp, ym, zp, zm;
};
__device__ __forceinline__ QNbr load_q_nbr(const double *__restrict__ Q, const CompactArgs &A, int x, int y, int z,
                                           int64_t cell)
{
    const int64_t sy = A.nx, sz = int64_t(A.nx) * A.ny;
    QNbr r;
    r.xp = Q[cell + (x + 1 < A.nx ? 1 : 0)];
    r.xm = Q[cell - (x > 0 ? 1 : 0)];
    r.yp = Q[A.N + cell + (y + 1 < A.ny ? sy : 0)];
    r.ym = Q[A.N + cell - (y > 0 ? sy : 0)];
    r.zp = Q[2 * A.N + cell + (z + 1 < A.nz ? sz : 0)];
    r.zm = Q[2 * A.N + cell - (z > 0 ? sz : 0)];
    return r;
}

__device__ __forceinline__ bool cell_coords(const CompactArgs &A, int &x, int &y, int &z, int64_t &cell)
{
    x = int(blockIdx.x * blockDim.x + threadIdx.x);
    y = int(blockIdx.y * blockDim.y + threadIdx.y);
    z = int(blockIdx.z);
    if (x >= A.nx || y >= A.ny) return false;
    cell = (int64_t(z) * A.ny + y) * A.nx + x;
    return true;
}

// FP16 storage: the block's largest |population - shift| per lattice goes
// to the written buffer's box entries (every block lies in one z-plane, so
// in one scale box); a block whose largest value exceeded the FP16 range
// at its scale (so that some value was clamped) is counted; the box's new
// exponent is stored by each of its blocks (the same value)
__device__ __forceinline__ void half_block_stats(const Half16 &h16, int b, int ef, int eg, float mf, float mg)
{
    __shared__ float smf[16], smg[16];  // one per wave, blocks up to 1024 threads
    for (int o = 32; o > 0; o >>= 1) {
        mf = fmaxf(mf, __shfl_xor(mf, o));
        mg = fmaxf(mg, __shfl_xor(mg, o));
    }
    const int t = threadIdx.y * blockDim.x + threadIdx.x;
    const int wv = t / 64;
    if ((t & 63) == 0) {
        smf[wv] = mf;
        smg[wv] = mg;
    }
    __syncthreads();
    if (t == 0) {
        const int nw = int(blockDim.x * blockDim.y) / 64;
        for (int i = 1; i < nw; ++i) {
            mf = fmaxf(mf, smf[i]);
            mg = fmaxf(mg, smg[i]);
        }
        atomicMax(&h16.amax_next[2 * b], __float_as_uint(mf));
        atomicMax(&h16.amax_next[2 * b + 1], __float_as_uint(mg));
        const uint32_t nsat = uint32_t(ldexpf(mf, ef) > 65504.0f) + uint32_t(ldexpf(mg, eg) > 65504.0f);
        if (nsat) atomicAdd(h16.ovf, nsat);
        h16.e_next[2 * b] = ef;
        h16.e_next[2 * b + 1] = eg;
    }
}

// equilibria and relaxation of a pulled cell in arithmetic type R;
// put(q, f', g') receives the post-collision populations
template <class R, class Put>
__device__ __forceinline__ void relax_cell(const R fv[NQ], const R gv[NQ], const MomentsR<R> &mo, const MacroR<R> &M,
                                           double dqx, double dqy, double dqz, const CollideParams &P, Put &&put)
{
    if constexpr (std::is_same<R, double>::value) {
        collide_cell_t<R>(fv, gv, mo, M, dqx, dqy, dqz, P, [&](auto qc, R fnew, R gnew) { put(qc, fnew, gnew); });
    } else {
        // FP32 equilibria; their sums would miss rho and E by the FP32
        // rounding of the coefficients, the same for similar cells
        // every step.  The rest direction's equilibria are rho and E
        // less the FP64 sums of the other 26, so that each cell's
        // equilibria carry its mass and energy; it is relaxed last,
        // which keeps only the two running sums live.
        const CollideCoeffsR<R> C = collide_coeffs_t<R>(mo, M, R(dqx), R(dqy), R(dqz), P);
        const R omega = C.omega;
        // rho and E as FP64 sums of the pulled values
        double rho_d = 0.0, e_d = 0.0;
        static_for<NQ>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            rho_d += double(fv[q]);
            e_d += double(gv[q]);
        });
        double sf = 0.0, sg = 0.0;
        static_for<NQ - 1>([&](auto pc) {
            constexpr int q = decltype(pc)::value + 1;
            const R fe = feq_of<q>(C), ge = geq_of<q>(C);
            sf += double(fe);
            sg += double(ge);
            put(std::integral_constant<int, q>{}, fv[q] + omega * (fe - fv[q]), gv[q] + omega * (ge - gv[q]));
        });
        const R fe0 = R(rho_d - sf), ge0 = R(e_d - sg);
        put(std::integral_constant<int, 0>{}, fv[0] + omega * (fe0 - fv[0]), gv[0] + omega * (ge0 - gv[0]));
    }
}

// Pass 2 of the shifted FP32 storage with FP32 arithmetic, in deviation
// form.  The populations are handled as their stored differences d = f - s
// from the rest equilibrium s (O(1e-2) of f), so that FP32 rounding applies
// to the differences, not to the populations:
//  - moments: FP64 sums of the pulled differences plus the shift's moments;
//    macroscopic fields, the gradient and the equilibrium coefficients in
//    FP64, as the FP64 collide computes them;
//  - f equilibria: with A, B, C the x, y, z factors of the product form and
//    A0, B0, C0 the shift's, A B C - A0 B0 C0 = (dA B + A0 dB) C + A0 B0 dC,
//    the factor differences taken in FP64 and the products in FP32;
//  - g equilibria: w_q (dE + c.a1 + (dS)/2), the differences of the Grad
//    coefficients from the shift's taken in FP64;
//  - relaxation d' = d + omega (d_eq - d) in FP32;
//  - the rest direction's equilibrium difference is the FP64 sum of the
//    pulled differences less the FP64 sum of the other 26 (for f and g),
//    so that each cell's equilibria carry its mass and energy exactly;
//  - the FP64 momentum residual of the 26 FP32 f equilibria goes, half and
//    half with opposite signs, to the pair c = +-e_a of each axis, so that
//    they carry the pulled momentum too (without it the rounding, alike in
//    neighbouring cells, drifts the velocity: 2e-6 after 100 steps against
//    4e-7 with it).
// the FP64 moments of the pulled differences of a cell (fv, gv: arrays or
// LDS rows of FP32 values) plus the shift's; their mass, energy and
// momentum sums kept apart for the residuals of the FP32 equilibria
struct F32Sums {
    double rho_d, e_d, jd[3];
};
template <class SF, class SG>
__device__ __forceinline__ void f32_moments(const SF &fv, const SG &gv, const DevRest &D, MomentsR<double> &mo,
                                            F32Sums &ds)
{
    accumulate_moments(fv, gv, mo);
    ds.rho_d = mo.rho;  // sums of the differences
    ds.e_d = mo.E;
    ds.jd[0] = mo.jx;
    ds.jd[1] = mo.jy;
    ds.jd[2] = mo.jz;
    mo.rho += D.mo[0];
    mo.jx += D.mo[1];
    mo.jy += D.mo[2];
    mo.jz += D.mo[3];
    mo.pxx += D.mo[4];
    mo.pyy += D.mo[5];
    mo.pzz += D.mo[6];
    mo.pxy += D.mo[7];
    mo.pxz += D.mo[8];
    mo.pyz += D.mo[9];
    mo.E += D.mo[10];
    mo.qx += D.mo[11];
    mo.qy += D.mo[12];
    mo.qz += D.mo[13];
}

// the equilibria in FP32 from the FP64 coefficients and the relaxation of
// the differences; put(q, f', g') receives the post-collision differences
template <class SF, class SG, class Put>
__device__ __forceinline__ void f32_relax(const SF &fv, const SG &gv, const MomentsR<double> &mo, const Macro &M,
                                          const F32Sums &ds, double dqx, double dqy, double dqz, const DevRest &D,
                                          const CollideParams &P, Put &&put)
{
    const double rho_d = ds.rho_d, e_d = ds.e_d;
    const double *jd = ds.jd;
    const CollideCoeffs C = collide_coeffs(mo, M, dqx, dqy, dqz, P);
    // factor and coefficient differences from the rest state (FP64, then FP32)
    float dA[3], Bf[3], dB[3], Cf[3], dC[3], A0f[3], B0f[3];
    for (int k = 0; k < 3; ++k) {
        dA[k] = float(C.rphx[k] - D.A0[k]);
        Bf[k] = float(C.phy[k]);
        dB[k] = float(C.phy[k] - D.B0[k]);
        Cf[k] = float(C.phz[k]);
        dC[k] = float(C.phz[k] - D.B0[k]);
        A0f[k] = float(D.A0[k]);
        B0f[k] = float(D.B0[k]);
    }
    const float dE = float(C.E - D.E0);
    const float a1x = float(C.a1x), a1y = float(C.a1y), a1z = float(C.a1z);
    float dtx[2], dty[2], dtz[2];
    for (int k = 0; k < 2; ++k) {
        dtx[k] = float(C.tx[k] - D.t0[k]);
        dty[k] = float(C.ty[k] - D.t0[k]);
        dtz[k] = float(C.tz[k] - D.t0[k]);
    }
    const float dxy = float(C.dxy), dxz = float(C.dxz), dyz = float(C.dyz);
    const float omega = float(C.omega);
    // the 26 moving directions' equilibrium differences, with FP64 sums of
    // their momentum
    float fe[NQ], ge[NQ];
    double sj[3] = {0.0, 0.0, 0.0};
    static_for<NQ - 1>([&](auto pc) {
        constexpr int q = decltype(pc)::value + 1;
        constexpr int cx = ev(q, 0), cy = ev(q, 1), cz = ev(q, 2);
        fe[q] = (dA[cx + 1] * Bf[cy + 1] + A0f[cx + 1] * dB[cy + 1]) * Cf[cz + 1] +
                (A0f[cx + 1] * B0f[cy + 1]) * dC[cz + 1];
        float gq = dE;
        if constexpr (cx == 1) gq = gq + a1x;
        if constexpr (cx == -1) gq = gq - a1x;
        if constexpr (cy == 1) gq = gq + a1y;
        if constexpr (cy == -1) gq = gq - a1y;
        if constexpr (cz == 1) gq = gq + a1z;
        if constexpr (cz == -1) gq = gq - a1z;
        float S = dtx[cx * cx] + dty[cy * cy];
        if constexpr (cx * cy == 1) S = S + dxy;
        if constexpr (cx * cy == -1) S = S - dxy;
        S = S + dtz[cz * cz];
        if constexpr (cx * cz == 1) S = S + dxz;
        if constexpr (cx * cz == -1) S = S - dxz;
        if constexpr (cy * cz == 1) S = S + dyz;
        if constexpr (cy * cz == -1) S = S - dyz;
        ge[q] = (gq + 0.5f * S) * float(weight(q));
        if constexpr (cx != 0) sj[0] += cx * double(fe[q]);
        if constexpr (cy != 0) sj[1] += cy * double(fe[q]);
        if constexpr (cz != 0) sj[2] += cz * double(fe[q]);
    });
    // Their momentum is the pulled momentum less the rest state's (zero)
    // in exact arithmetic; the FP32 rounding of the 26 products leaves a
    // residual that the same rounding repeats in neighbouring cells, so the
    // velocity would drift coherently.  The residual of each axis goes to
    // that axis's pair of directions c = +-e_a (half each, opposite signs:
    // mass and the second moments are unchanged).
    static_for<3>([&](auto ac) {
        constexpr int a = decltype(ac)::value;
        constexpr int qp = a == 0 ? qof(1, 0, 0) : (a == 1 ? qof(0, 1, 0) : qof(0, 0, 1));
        constexpr int qm = kBounce[qp];
        const float h = float(0.5 * (jd[a] - sj[a]));
        fe[qp] = fe[qp] + h;
        fe[qm] = fe[qm] - h;
    });
    double sf = 0.0, sg = 0.0;
    static_for<NQ - 1>([&](auto pc) {
        constexpr int q = decltype(pc)::value + 1;
        sf += double(fe[q]);
        sg += double(ge[q]);
        put(std::integral_constant<int, q>{}, fv[q] + omega * (fe[q] - fv[q]), gv[q] + omega * (ge[q] - gv[q]));
    });
    const float fe0 = float(rho_d - sf), ge0 = float(e_d - sg);
    put(std::integral_constant<int, 0>{}, fv[0] + omega * (fe0 - fv[0]), gv[0] + omega * (ge0 - gv[0]));
}

__device__ __forceinline__ void store_agent(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_agent(double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every memory access of the wave issued so far has completed
__device__ __forceinline__ void drain_wave()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

CompactArgs make_args(const mrb_level *L)
{
    CompactArgs A{};
    A.nx = L->ncell[0];
    A.ny = L->ncell[1];
    A.nz = L->ncell[2];
    for (int d = 0; d < 3; ++d) A.per[d] = L->periodic[d];
    A.N = L->total_cells;
    A.cs = 2 * A.N;
    for (int n = 0; n < 6; ++n) A.bc[n] = L->bc.bc_type[n];
    A.bcpack = 0;
    for (int n = 0; n < 6; ++n) A.bcpack |= uint32_t(A.bc[n] & 15) << (4 * n);
    // bytes of one cell's (f_q, g_q) pair
    const int64_t cell_bytes = L->storage == MRB_STORAGE_F64 ? 16 : (L->storage == MRB_STORAGE_F32_SHIFTED ? 8 : 4);
    A.fast_ok = A.N * cell_bytes < (int64_t(1) << 32) ? 1 : 0;
    return A;
}

ShiftTab shift_tab(const mrb_level *L)
{
    ShiftTab t{};
    if (L->storage != MRB_STORAGE_F64) {
        const int rep[4] = {0, 1, 7, 19};
        for (int k = 0; k < 4; ++k) {
            t.fk[k] = L->fshift[rep[k]];
            t.gk[k] = L->gshift[rep[k]];
        }
    }
    return t;
}

// the boundary floor of the FP16 box maxima: |f_eq - shift| and
// |g_eq - shift| of the inlet state (for a Channel or Parabolic profile the
// reference speed bounds the profile) and of the pressure faces' state at
// rest and at their g velocity
void f16_floors(const mrb_level *L, float &ff, float &fg)
{
    double mf = 0.0, mg = 0.0;
    const BCDev &d = L->bcdev;
    auto take = [&](const double *fv, const double *gv) {
        for (int q = 0; q < NQ; ++q) {
            mf = std::max(mf, std::fabs(fv[q] - L->fshift[q]));
            mg = std::max(mg, std::fabs(gv[q] - L->gshift[q]));
        }
    };
    bool velocity = false;
    for (int n = 0; n < 6; ++n) velocity = velocity || L->bc.bc_type[n] == MRB_BC_VELOCITY;
    if (velocity) {
        if (d.prof.kind) {
            const VelProfile &P = d.prof;
            double fv[NQ], gv[NQ];
            for (int dir = 0; dir < 3; ++dir)
                for (int sgn = -1; sgn <= 1; sgn += 2) {
                    double v[3] = {0.0, 0.0, 0.0};
                    v[dir] = sgn * P.vref;
                    for (int q = 0; q < NQ; ++q) {
                        fv[q] = set_equilibrium_value(P.rho, v, P.R * P.T, q);
                        gv[q] = thermal_g_equilibrium(P.rho, v, P.T, P.R, P.gamma, q);
                    }
                    take(fv, gv);
                }
        } else {
            take(d.fval, d.gval);
        }
    }
    if (d.pdir >= 0) {
        const double zero[3] = {0.0, 0.0, 0.0};
        for (int q = 0; q < NQ; ++q) {
            mf = std::max(mf, std::fabs(set_equilibrium_value(d.prho, zero, d.prt, q) - L->fshift[q]));
            if (kEV[q][d.pdir] != 0) mg = std::max(mg, std::fabs(d.pgval[q] - L->gshift[q]));
        }
    }
    ff = float(mf);
    fg = float(mg);
}

DevRest dev_rest(const mrb_level *L)
{
    DevRest d{};
    if (L->storage != MRB_STORAGE_F32_SHIFTED) return d;
    const double R = kAirMolarMass / (L->phys_set ? L->phys.m_bar : kAirMolarMass);
    const double gamma = L->phys_set ? L->phys.adiabatic_exponent : 5.0 / 3.0;
    const double rho0 = L->shift_rho0, T0 = L->shift_T0, rt = R * T0;
    // the factors of set_equilibrium_value at u = 0 (the f shift is
    // ((rho0 phi_x) phi_y) phi_z of these)
    for (int c = -1; c <= 1; ++c) {
        const double pxx = 0.0 * 0.0 + rt;
        const double phi = c * 0.5 * 0.0 + iabs(c) * (1.50 * pxx - 1.0) - pxx + 1.0;
        d.B0[c + 1] = phi;
        d.A0[c + 1] = rho0 * phi;
    }
    // the Grad coefficients of thermal_g_equilibrium at u = 0
    const double cv = R / (gamma - 1.0);
    const double E = rho0 * (2.0 * cv * T0 + 0.0 * 0.0 + 0.0 * 0.0 + 0.0 * 0.0);
    const double energy = E / (2.0 * rho0);
    const double Tv = (0.50 / cv) * ((E / rho0) - 0.0 * 0.0 + 0.0 * 0.0 + 0.0 * 0.0);
    const double p = rho0 * R * Tv;
    const double h = energy + (p / rho0);
    const double rxx = 2.0 * rho0 * 0.0 * 0.0 * (h + p / rho0) + 2.0 * p * h;
    const double inv = 1.0 / kTheta0;
    const double a2xx = (rxx - E * 1.0 * kTheta0) * inv * inv;
    d.E0 = E;
    d.t0[0] = (0 - kTheta0) * a2xx;
    d.t0[1] = (1 - kTheta0) * a2xx;
    MomentsR<double> m;
    accumulate_moments(L->fshift, L->gshift, m);
    const double mo[14] = {m.rho, m.jx, m.jy, m.jz, m.pxx, m.pyy, m.pzz, m.pxy, m.pxz, m.pyz, m.E, m.qx, m.qy, m.qz};
    for (int k = 0; k < 14; ++k) d.mo[k] = mo[k];
    return d;
}

Half16 half16_of(mrb_level *L)
{
    Half16 h{};
    if (L->storage == MRB_STORAGE_F16_SCALED) {
        h.e_cur = L->d_e16[L->cur];
        h.e_next = L->d_e16[1 - L->cur];
        h.amax_cur = L->d_amax16[L->cur];
        h.amax_next = L->d_amax16[1 - L->cur];
        h.ovf = L->d_ovf16;
        f16_floors(L, h.floor_f, h.floor_g);
    }
    return h;
}

// blocks of a kernel that the GPU holds at once (occupancy x CUs): the
// z-sweeps wait on each other and need every block resident; they are
// launched only when the occupancy calculation says so (their waits are
// bounded, so a block that is not resident after all turns into NaN
// results and a fault count, not a hang)
int resident_blocks(const void *kernel, int threads, int &fit)
{
    static std::mutex mu;
    static std::map<std::pair<int, const void *>, int> cache;  // (device, kernel) -> blocks
    int dev = 0;
    MRB_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    const auto key = std::make_pair(dev, kernel);
    const auto it = cache.find(key);
    if (it != cache.end()) {
        fit = it->second;
        return MRB_OK;
    }
    int per_cu = 0, cus = 0;
    MRB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    MRB_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0));
    fit = per_cu * cus;
    cache[key] = fit;
    return MRB_OK;
}

// the inlet-profile lookups and the pressure ghosts are compiled only into
// the kernels of levels that have them
int bcx_of(const mrb_level *L)
{
    return (L->bcdev.prof.kind ? kBcxProfile : 0) | (L->bcdev.pdir >= 0 ? kBcxPressure : 0);
}

}  // namespace
}  // namespace mrb
