// The two-pass step of the compact layout on tiles of consecutive cells.
//
// A tile is 256 (FP32 storage: 128) consecutive cells of a z-plane, whatever
// the row length: on 301-cell rows 256x1 blocks leave 41 % of their lanes
// idle, on 24-cell rows 91 %.  A tile's z is the same for all its lanes, so
// the pull's loads take a scalar base and a 32-bit offset, and they are
// issued together with the load of the stream mask: lanes next to solid cells
// or walls load those sources again (pull_settle).
//
// k_step: both passes of an FP64 level in one launch.  Pass 1 (Q_corr of the
// post-stream state) and pass 2 (collide, which needs the six face
// neighbours' Q_corr) pull the same 54 populations.  As two launches the
// second pull finds nothing left of the first one in the caches: at 256^3
// 22.9 GB move per step at the HBM rate.  Here the tiles of both passes are
// handed out from one list in which pass 2 follows pass 1 at a fixed distance
// (a plane and the tiles in flight), so that the second pull hits the 256 MB
// memory-side cache; its loads are non-temporal, since nothing reads the
// values again.  256^3: 4.30 -> 3.24 ms per step; 301x150x131: 1.95 ->
// 1.19 ms.  The same traffic through the fabric (22.6 GB) then moves at 7 TB/s,
// which is what bounds it: 24 % fewer vector instructions changed nothing.
// Shifted FP32 storage stays on two launches: pass 2 holds twice the
// registers of pass 1, so in one kernel pass 1 runs at half its occupancy,
// and with half the bytes per wave that costs more than the cache saves
// (320^3: 4.74 ms against 4.46); scaled FP16 likewise (256^3: 1.77 ms against
// 1.68 for the step alone).
//
// Order and progress: a block takes the next entry of the list from an atomic
// counter.  A pass-2 tile waits for the pass-1 tiles it reads Q_corr from;
// those have lower list positions, so they were taken before by blocks that
// are running, and a pass-1 tile waits for nothing.  Every wait therefore
// ends, however many blocks the GPU holds and whatever else it runs.  (The
// waits are bounded all the same; past the limit the tile counts a fault, which
// mrb_step_faults reports, and writes NaN.)
//
// Q_corr crosses XCDs, whose L2s are not coherent: it is written and read by
// agent-scope accesses, and a tile's flag (the launch's epoch) is stored
// after the tile's Q_corr writes have completed.  Q_x only leaves the block
// for the tile's two end cells.  The block that takes the launch's last entry
// resets the list and advances the epoch, so a captured launch can be replayed;
// the blocks still at work keep the epoch they took with their entry.
#include "compact_cell.h"

namespace mrb {
namespace {

constexpr int kStepTile = 256;
// FP32 storage: 128-cell tiles (320^3: 4.46 ms against 4.56 with 256)
constexpr int kF32Tile = 128;
// k_step takes FP64 levels of at least this many cells: below, both passes'
// populations stay in the memory-side cache anyway (2^18 cells are 113 MB) and
// the work list's counter and flags only add to the step.  Periodic boxes, us
// per step in one launch / with the passes apart: 24^3 14.4 / 12.4, 40^3 25.9 /
// 18.1, 56^3 52.4 / 43.8, 64^3 62.3 / 62.8, 72^3 91.9 / 91.8, 80^3 118 / 126,
// 96^3 188 / 212, 128^3 414 / 523; thin ones cross later (660x123x4 83.5 / 80.8).
constexpr int64_t kListCells = 1 << 18;
// pass-1 tiles ahead of pass 2 besides a plane: the blocks 256 CUs hold at
// two each, so that the tiles waited for are usually done (256^3: 3.29 ms with
// 128, 3.23 with 256 to 1024, 3.50 with 2048, which leaves the cache)
constexpr uint32_t kListAhead = 512;
// a block's lanes watch the tiles its rows reach
constexpr int kListRow = 32000;
constexpr uint32_t kStepSpinLimit = 1u << 22;

// n / d for 32-bit n by a multiplication (round-up method)
struct FastDiv {
    uint32_t d, m, s1, s2;
    explicit FastDiv(uint32_t d_) : d(d_)
    {
        uint32_t l = 0;
        while (l < 32 && (uint64_t(1) << l) < d) ++l;
        m = uint32_t((((uint64_t(1) << l) - d) << 32) / d + 1);
        s1 = l < 1 ? l : 1;
        s2 = l > 0 ? l - 1 : 0;
    }
    __device__ __forceinline__ uint32_t div(uint32_t n) const
    {
        const uint32_t t = __umulhi(m, n);
        return (t + ((n - t) >> s1)) >> s2;
    }
};

// the tiles of a level
struct TileArgs {
    uint32_t nxy;  // cells of a z-plane
    uint32_t tpp;  // tiles of a z-plane
    FastDiv by_tpp, by_nx;
};

// the work list of k_step
struct ListArgs {
    uint32_t ntiles;  // tpp * nz
    uint32_t lag;     // pass-1 tiles ahead of pass 2, > tpp (or ntiles)
    uint32_t wrow;    // tiles a row spans: a tile's y neighbours lie within -+ wrow tiles
    unsigned long long *counter;  // launches so far (high half), list entries taken (low half)
    uint32_t *flags;              // per tile: launch whose Q_corr it holds
    uint32_t *fault;              // waits that ran out
};

__device__ __forceinline__ uint32_t load_agent_u32(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent_u32(uint32_t *p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Arithmetic of pass 2
enum StepArith { kStepF64 = 0, kStepF32Dev = 1, kStepH32 = 2 };

// list entry t: pass-1 tiles 0 .. lag-1, then pass-2 tile j and pass-1 tile
// lag + j in turn, then the remaining pass-2 tiles; returns the tile
__device__ __forceinline__ uint32_t list_entry(uint32_t t, const ListArgs &S, bool &pass2)
{
    pass2 = false;
    if (t < S.lag) return t;
    const uint32_t u = t - S.lag, both = 2u * (S.ntiles - S.lag);
    if (u < both) {
        pass2 = (u & 1u) == 0u;
        return pass2 ? u >> 1 : S.lag + (u >> 1);
    }
    pass2 = true;
    return (S.ntiles - S.lag) + (u - both);
}

// the cell a lane of a tile works on; lanes past the plane's end repeat its
// last cell's work and store nothing
struct TileCell {
    int x, y, z;
    uint32_t r;  // tile within the plane
    int64_t cell;
    bool in;
    template <int TILE>
    __device__ __forceinline__ static TileCell of(uint32_t tile, const CompactArgs &A, const TileArgs &G)
    {
        TileCell c;
        c.z = int(G.by_tpp.div(tile));
        c.r = tile - uint32_t(c.z) * G.tpp;
        const uint32_t k = c.r * TILE + threadIdx.x, c2 = min(k, G.nxy - 1u);
        c.in = k < G.nxy;
        c.y = int(G.by_nx.div(c2));
        c.x = int(c2 - uint32_t(c.y) * uint32_t(A.nx));
        c.cell = int64_t(c.z) * G.nxy + c2;
        return c;
    }
};

// pass 1 of a tile: Q_corr of the post-stream state.  LISTED: read by other
// blocks of the same launch (agent-scope stores; Q_x of the end cells only)
template <class T, int BCX, bool LISTED>
__device__ __forceinline__ void pass1_tile(
    const T *__restrict__ f, const uint32_t *__restrict__ mask, double *Q, const CompactArgs &A, const BCDev &bc,
    const ShiftTab &sh, const Half16 &h16, const CollideParams &P, const TileCell &c)
{
    if constexpr (kIsHalf<T>) {
        // box maxima of the buffer pass 2 writes, cleared by each slab's first tile
        if (c.z % kScaleSlab == 0 && c.r == 0 && threadIdx.x < 2)
            h16.amax_next[2 * (c.z / kScaleSlab) + int(threadIdx.x)] = 0u;
    }
    T rf[NQ], rg[NQ];
    const uint32_t m0 = mask[c.cell];
    pull_ahead<T, false>(f, A, c.x, c.y, c.z, rf, rg);
    // (a solid cell pulls as if all its sources were fluid)
    const uint32_t m = (m0 & 1u) ? m0 : (m0 | kAllQ);
    const PullBits pb = pull_settle<BCX, T, false>(f, A, c.x, c.y, c.z, c.cell, m, rf, rg);
    double fv[NQ], gv[NQ];
    pull_finish<BCX, T, double>(f, A, bc, sh, h16, c.x, c.y, c.z, m, pb, rf, rg, fv, gv);
    double rho, jx, jy, jz, E;
    accumulate_q_moments(fv, gv, rho, jx, jy, jz, E);
    const Macro M = macro_from(rho, jx, jy, jz, E, P);
    if (c.in && (m0 & 1u)) {
        if constexpr (LISTED) {
            if (threadIdx.x == 0 || threadIdx.x == kStepTile - 1) store_agent(&Q[c.cell], M.Qx);
            store_agent(&Q[A.N + c.cell], M.Qy);
            store_agent(&Q[2 * A.N + c.cell], M.Qz);
        } else {
            Q[c.cell] = M.Qx;
            Q[A.N + c.cell] = M.Qy;
            Q[2 * A.N + c.cell] = M.Qz;
        }
    }
}

// pass 2 of a tile: stream + collide.  LISTED (FP64 arithmetic): waits for
// the flags of the pass-1 tiles it reads Q_corr from, while its pull is in
// flight; Q_x reaches the x neighbours through LDS, since with FP64 arithmetic
// pass 2's own moments give it bit for bit as pass 1's do
template <class T, int BCX, int ARITH, bool LISTED>
__device__ __forceinline__ void pass2_tile(
    const T *__restrict__ f, T *__restrict__ fo, const uint32_t *__restrict__ mask, double *Q, const CompactArgs &A,
    const BCDev &bc, const ShiftTab &sh, const Half16 &h16, const DevRest &D, const CollideParams &P,
    const TileArgs &G, const TileCell &c, const ListArgs &S, uint32_t epoch)
{
    static_assert(!LISTED || (ARITH == kStepF64 && !kIsHalf<T>), "work list: FP64 arithmetic only");
    constexpr bool kDev = ARITH == kStepF32Dev;
    using R = std::conditional_t<ARITH == kStepF64, double, float>;   // pulled values
    using RM = std::conditional_t<ARITH == kStepH32, float, double>;  // their moments
    T *const go = fo + 1;
    const uint32_t tid = threadIdx.x;
    const int x = c.x, y = c.y, z = c.z;
    const int64_t cell = c.cell;
    uint32_t watch = 0u, seen = epoch;
    if constexpr (LISTED) {
        // lane k watches one tile: the row neighbours in the plane, then the
        // tile's own position in the planes beside
        const uint32_t tile = uint32_t(z) * G.tpp + c.r;
        const uint32_t lo = c.r > S.wrow ? c.r - S.wrow : 0u, hi = min(c.r + S.wrow, G.tpp - 1u);
        const uint32_t nrow = hi - lo + 1u;
        watch = uint32_t(z) * G.tpp + lo + min(tid, nrow - 1u);
        if (tid == nrow && z > 0) watch = tile - G.tpp;
        if (tid == nrow + 1u && z + 1 < A.nz) watch = tile + G.tpp;
        seen = load_agent_u32(&S.flags[watch]);
    }
    const uint32_t m0 = mask[cell];
    T rf[NQ], rg[NQ];
    pull_ahead<T, true>(f, A, x, y, z, rf, rg);
    bool poisoned = false;
    // Q_corr of the neighbours, clamped into the domain (a value past a face
    // is loaded but not used)
    const int64_t sy = A.nx, sz = G.nxy;
    double qxp, qxm, qyp, qym, qzp, qzm;
    if constexpr (LISTED) {
        for (uint32_t it = 0; !__syncthreads_and(seen == epoch); ++it) {
            if (it > kStepSpinLimit) {
                poisoned = true;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
            seen = load_agent_u32(&S.flags[watch]);
        }
        qxm = qxp = 0.0;
        if (tid == 0) qxm = load_agent(&Q[cell - (x > 0 ? 1 : 0)]);
        if (tid == kStepTile - 1) qxp = load_agent(&Q[cell + (x + 1 < A.nx ? 1 : 0)]);
        qyp = load_agent(&Q[A.N + cell + (y + 1 < A.ny ? sy : 0)]);
        qym = load_agent(&Q[A.N + cell - (y > 0 ? sy : 0)]);
        qzp = load_agent(&Q[2 * A.N + cell + (z + 1 < A.nz ? sz : 0)]);
        qzm = load_agent(&Q[2 * A.N + cell - (z > 0 ? sz : 0)]);
    } else {
        const QNbr q = load_q_nbr(Q, A, x, y, z, cell);
        qxp = q.xp;
        qxm = q.xm;
        qyp = q.yp;
        qym = q.ym;
        qzp = q.zp;
        qzm = q.zm;
    }
    const bool fluid = (m0 & 1u) != 0;
    const uint32_t m = fluid ? m0 : (m0 | kAllQ);
    const PullBits pb = pull_settle<BCX, T, true>(f, A, x, y, z, cell, m, rf, rg);
    R fv[NQ], gv[NQ];
    pull_finish<BCX, T, R, kDev>(f, A, bc, sh, h16, x, y, z, m, pb, rf, rg, fv, gv);
    MomentsR<RM> mo;
    F32Sums ds;
    if constexpr (kDev)
        f32_moments(fv, gv, D, mo, ds);
    else
        accumulate_moments(fv, gv, mo);
    const MacroR<RM> M = macro_from_t<RM>(mo.rho, mo.jx, mo.jy, mo.jz, mo.E, P);
    if constexpr (LISTED) {
        __shared__ double qx[kStepTile];
        qx[tid] = M.Qx;
        __syncthreads();
        if (tid > 0) qxm = qx[tid - 1];
        if (tid < kStepTile - 1) qxp = qx[tid + 1];
    }
    // gradient(): neighbour inside the domain box and fluid
    const bool xp = x < A.nx - 1 && ((m0 >> 2) & 1u), xm = x > 0 && ((m0 >> 1) & 1u);
    const bool yp = y < A.ny - 1 && ((m0 >> 4) & 1u), ym = y > 0 && ((m0 >> 3) & 1u);
    const bool zp = z < A.nz - 1 && ((m0 >> 6) & 1u), zm = z > 0 && ((m0 >> 5) & 1u);
    double dqx = one_sided_gradient(xp, xm, xp ? qxp : 0.0, M.Qx, xm ? qxm : 0.0, P.inv_dx[0]);
    const double dqy = one_sided_gradient(yp, ym, yp ? qyp : 0.0, M.Qy, ym ? qym : 0.0, P.inv_dx[1]);
    const double dqz = one_sided_gradient(zp, zm, zp ? qzp : 0.0, M.Qz, zm ? qzm : 0.0, P.inv_dx[2]);
    if (poisoned) {
        // (counted here: within the wait's loop it cost 0.5 % of the step)
        dqx = __builtin_nan("");
        if (tid == 0) atomicAdd(S.fault, 1u);
    }
    float mf = 0.0f, mg = 0.0f;
    int ef = 0, eg = 0;
    if constexpr (kIsHalf<T>) {
        // scales of the written buffer from the read buffer's box maxima
        const int b = z / kScaleSlab;
        ef = f16_exponent(f16_pull_max(h16.amax_cur, b, 0, A.nz, A.per[2], h16.floor_f));
        eg = f16_exponent(f16_pull_max(h16.amax_cur, b, 1, A.nz, A.per[2], h16.floor_g));
    }
    if (c.in && fluid) {
        const float scf = ldexpf(1.0f, ef), scg = ldexpf(1.0f, eg);
        const float lif = ldexpf(65504.0f, -ef), lig = ldexpf(65504.0f, -eg);
        auto put = [&](auto qc, auto fnew, auto gnew) {
            constexpr int q = decltype(qc)::value;
            const int64_t e = int64_t(q) * A.cs + cell * kCellStride<T>;
            if constexpr (kIsHalf<T>)
                store_pair(fo, go, e, to_half(fnew, decltype(fnew)(sh.f(q)), scf, lif, mf),
                           to_half(gnew, decltype(gnew)(sh.g(q)), scg, lig, mg));
            else if constexpr (kDev)
                store_pair(fo, go, e, fnew, gnew);
            else
                store_pair(fo, go, e, narrow<T>(fnew, sh.f(q)), narrow<T>(gnew, sh.g(q)));
        };
        if constexpr (kDev)
            f32_relax(fv, gv, mo, M, ds, dqx, dqy, dqz, D, P, put);
        else
            relax_cell<R>(fv, gv, mo, M, dqx, dqy, dqz, P, put);
    } else if (c.in) {
        // solid cell: the stream leaves the -1 sentinel (LBM.cpp:565); FP16
        // storage holds 0 there (downloads return the sentinel)
        static_for<NQ>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int64_t e = int64_t(q) * A.cs + cell * kCellStride<T>;
            if constexpr (kIsHalf<T>)
                store_pair(fo, go, e, T(0.0f), T(0.0f));
            else
                store_pair(fo, go, e, narrow<T>(-1.0, sh.f(q)), narrow<T>(-1.0, sh.g(q)));
        });
    }
    if constexpr (kIsHalf<T>) half_block_stats(h16, z / kScaleSlab, ef, eg, mf, mg);
}

// both passes, FP64 storage
template <int BCX>
__global__ void __launch_bounds__(kStepTile, 2) k_step(
    const double *__restrict__ f, double *__restrict__ fo, const uint32_t *__restrict__ mask, double *Q,
    CompactArgs A, BCDev bc, ShiftTab sh, CollideParams P, TileArgs G, ListArgs S)
{
    __shared__ uint64_t taken;
    if (threadIdx.x == 0) {
        // the block that takes the launch's last entry moves the counter on
        const unsigned long long t = atomicAdd(S.counter, 1ull);
        if (uint32_t(t) == 2u * S.ntiles - 1u) atomicAdd(S.counter, (1ull << 32) - 2ull * S.ntiles);
        taken = t;
    }
    __syncthreads();
    const uint32_t epoch = uint32_t(__builtin_amdgcn_readfirstlane(int(taken >> 32))) + 1u;
    bool pass2;
    const uint32_t tile = list_entry(uint32_t(__builtin_amdgcn_readfirstlane(int(taken))), S, pass2);
    const TileCell c = TileCell::of<kStepTile>(tile, A, G);
    if (pass2) {
        pass2_tile<double, BCX, kStepF64, true>(f, fo, mask, Q, A, bc, sh, Half16{}, DevRest{}, P, G, c, S, epoch);
        return;
    }
    pass1_tile<double, BCX, true>(f, mask, Q, A, bc, sh, Half16{}, P, c);
    drain_wave();
    __syncthreads();
    if (threadIdx.x == 0) store_agent_u32(&S.flags[tile], epoch);
}

// the passes apart
template <class T, int BCX, int TILE>
__global__ void __launch_bounds__(TILE) k_qpass_tile(
    const T *__restrict__ f, const uint32_t *__restrict__ mask, double *__restrict__ Q, CompactArgs A, BCDev bc,
    ShiftTab sh, Half16 h16, CollideParams P, TileArgs G)
{
    pass1_tile<T, BCX, false>(f, mask, Q, A, bc, sh, h16, P, TileCell::of<TILE>(blockIdx.x, A, G));
}
template <class T, int BCX, int ARITH, int TILE>
__global__ void __launch_bounds__(TILE, 2) k_collide_tile(
    const T *__restrict__ f, T *__restrict__ fo, const uint32_t *__restrict__ mask, double *__restrict__ Q,
    CompactArgs A, BCDev bc, ShiftTab sh, Half16 h16, DevRest D, CollideParams P, TileArgs G)
{
    pass2_tile<T, BCX, ARITH, false>(f, fo, mask, Q, A, bc, sh, h16, D, P, G,
                                     TileCell::of<TILE>(blockIdx.x, A, G), ListArgs{}, 0u);
}
// scaled FP16 storage with FP32 arithmetic, held to 128 registers: four
// waves per SIMD (with a profile inlet one value spills: 160x80x80 duct 138 us
// per step against 214 on row blocks without the bound)
template <class T, int BCX, int ARITH, int TILE>
__global__ void __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(4))) k_collide_tile_w4(
    const T *__restrict__ f, T *__restrict__ fo, const uint32_t *__restrict__ mask, double *__restrict__ Q,
    CompactArgs A, BCDev bc, ShiftTab sh, Half16 h16, DevRest D, CollideParams P, TileArgs G)
{
    pass2_tile<T, BCX, ARITH, false>(f, fo, mask, Q, A, bc, sh, h16, D, P, G,
                                     TileCell::of<TILE>(blockIdx.x, A, G), ListArgs{}, 0u);
}

// both passes in one launch
bool one_launch(const mrb_level *L)
{
    return L->storage == MRB_STORAGE_F64 && L->total_cells >= kListCells && L->ncell[0] <= kListRow;
}

template <class T, int BCX, int ARITH>
int launch(mrb_level *L, hipStream_t s, hipEvent_t *ev)
{
    const CompactArgs A = make_args(L);
    const ShiftTab sh = shift_tab(L);
    const Half16 h16 = half16_of(L);
    const T *f = (const T *)L->pop[0][L->cur];
    T *fo = (T *)L->pop[0][1 - L->cur];
    constexpr int TILE = std::is_same<T, float>::value ? kF32Tile : kStepTile;
    const uint32_t nxy = uint32_t(A.nx) * uint32_t(A.ny), tpp = tiles_per_plane(A.nx, A.ny, TILE);
    const uint32_t ntiles = tpp * uint32_t(A.nz);
    const TileArgs G{nxy, tpp, FastDiv(tpp), FastDiv(uint32_t(A.nx))};
    if (ev) MRB_HIP(hipEventRecord(ev[0], s));
    if constexpr (std::is_same<T, double>::value) {
        if (one_launch(L)) {
            const uint32_t lag = std::min(ntiles, tpp + 1u + kListAhead);
            const ListArgs S{ntiles, lag, uint32_t(A.nx + kStepTile - 1) / kStepTile, L->d_step_counter,
                             L->d_step_flags, L->d_sweep_fault};
            k_step<BCX><<<2u * ntiles, kStepTile, 0, s>>>(f, fo, L->d_mask, L->d_q, A, L->bcdev, sh, L->cp, G, S);
            MRB_HIP(hipGetLastError());
            if (ev) MRB_HIP(hipEventRecord(ev[1], s));
            return MRB_OK;
        }
    }
    k_qpass_tile<T, BCX, TILE><<<ntiles, TILE, 0, s>>>(f, L->d_mask, L->d_q, A, L->bcdev, sh, h16, L->cp, G);
    MRB_HIP(hipGetLastError());
    if (ev) MRB_HIP(hipEventRecord(ev[1], s));
    if constexpr (ARITH == kStepH32)
        k_collide_tile_w4<T, BCX, ARITH, TILE><<<ntiles, TILE, 0, s>>>(f, fo, L->d_mask, L->d_q, A, L->bcdev, sh, h16,
                                                                      DevRest{}, L->cp, G);
    else
        k_collide_tile<T, BCX, ARITH, TILE><<<ntiles, TILE, 0, s>>>(f, fo, L->d_mask, L->d_q, A, L->bcdev, sh, h16,
                                                                   dev_rest(L), L->cp, G);
    MRB_HIP(hipGetLastError());
    if (ev) MRB_HIP(hipEventRecord(ev[2], s));
    return MRB_OK;
}

template <class T, int ARITH>
int launch_bcx(mrb_level *L, hipStream_t s, hipEvent_t *ev)
{
    const int bcx = bcx_of(L);
    bool x_only = true;  // no VELOCITY face but x-lo
    for (int n = 1; n < 6; ++n) x_only = x_only && L->bc.bc_type[n] != MRB_BC_VELOCITY;
    if (bcx == kBcxProfile && x_only) return launch<T, kBcxProfile | kBcxProfileX, ARITH>(L, s, ev);
    if constexpr (ARITH == kStepF64) {
        if (bcx == kBcxPressure) return launch<T, kBcxPressure, ARITH>(L, s, ev);
        if (bcx == (kBcxProfile | kBcxPressure)) return launch<T, kBcxProfile | kBcxPressure, ARITH>(L, s, ev);
    } else if (bcx & kBcxPressure) {
        return set_error(MRB_E_UNSUPPORTED, "the FP32-arithmetic collide has no PRESSURE faces");
    }
    return bcx == kBcxProfile ? launch<T, kBcxProfile, ARITH>(L, s, ev) : launch<T, 0, ARITH>(L, s, ev);
}

}  // namespace

int compact_tile_step(mrb_level *L, bool fp32_collide, hipStream_t s, hipEvent_t *ev)
{
    if (L->storage == MRB_STORAGE_F64) return launch_bcx<double, kStepF64>(L, s, ev);
    if (L->storage == MRB_STORAGE_F32_SHIFTED)
        return fp32_collide ? launch_bcx<float, kStepF32Dev>(L, s, ev) : launch_bcx<float, kStepF64>(L, s, ev);
    return fp32_collide ? launch_bcx<_Float16, kStepH32>(L, s, ev) : launch_bcx<_Float16, kStepF64>(L, s, ev);
}

const char *compact_tile_kernels(const mrb_level *L, bool fp32_collide)
{
    if (one_launch(L)) return "k_step";
    return fp32_collide && L->storage == MRB_STORAGE_F16_SCALED ? "k_qpass_tile+k_collide_tile_w4"
                                                                : "k_qpass_tile+k_collide_tile";
}

}  // namespace mrb
