// Launch interface of the large-step kernels.
//
// Every kernel works on a batch of members (independent domains of possibly
// different shapes, one precision per batch). The batch keeps a device array
// of MemberArgs (grid, field pointers, step parameters) and, per launch
// shape, a block map: entry b of the map names the member and the member-local
// work tile of workgroup b. One launch therefore covers every member of the
// batch, and the map order decides which XCD runs which tiles.
#pragma once

#include "nimbus_internal.hpp"

#include <string>
#include <vector>

namespace nimbus
{

struct TimedLaunch
{
    const char* name;
    hipEvent_t start, stop;
};

struct Launcher
{
    hipStream_t stream = nullptr;
    bool timing = false;
    std::vector<TimedLaunch>* pending = nullptr;
    std::vector<hipEvent_t>* event_pool = nullptr;
    std::uint64_t* launches = nullptr;
    hipError_t error = hipSuccess;

    hipEvent_t take_event();
    void begin(const char* name, hipEvent_t& a);
    void end(const char* name, hipEvent_t a);
};

// Device field set of one member (precision-erased pointers). rho' has a
// second buffer: acoustic substep s reads buffer s & 1 and writes (s + 1) & 1.
struct DevFields
{
    void *u, *v, *w, *rp, *pp, *th, *qv, *qc, *qr;       // prognostic state (rho, p as perturbations)
    void *u2, *v2, *w2, *rp2;                            // Heun predictor u, v, w; second rho' buffer
    void *mfx, *mfy, *mfz, *rb;                          // retained mass fluxes, rho' at step begin
    void *k1u, *k1v, *k1w;                               // Heun stage-1 tendencies
    void *tth, *tqv, *tqc, *tqr;                         // transported scalars before microphysics
    void* flux[12];                                      // per scalar: x, y, z face fluxes (7 alias dead slots)
    float *rl_qv, *rl_qc, *rl_qr;                        // PD limiter factors
    float *rad_w, *rad_e, *rad_s, *rad_n;                // KW78 radiative stashes
    double* rain;                                        // accumulated surface rain [ny][nx]
    double* base;                                        // kBaseCount * nz FP64 profiles
    double* diag;                                        // kDiagBlocksPerMember * kDiagValues partials + result
    double* sponge_lat;                                  // lateral sponge factor by distance to the nearest face
    double* clock;                                       // microphysics subcycle clock: elapsed, step, limit bits
};

struct StepParams
{
    double dt;          // large step
    double dts;         // acoustic substep
    double mf_weight;   // retained mass-flux weight per substep (dts / dt in the large step)
    int substeps;
    int acoustic_mode;
    double hevi_alpha;  // (1 + beta) / 2
    double coriolis_f;
    int bc_west, bc_east, bc_south, bc_north, bc_bottom, bc_top;
    int kessler_sub;    // microphysics subcycle launches per large step
    int kessler_adaptive; // subcycle lengths follow the state's sedimentation limit (device clock)
    int sponge;         // Rayleigh sponges on
    int sponge_lateral; // lateral band width (cells)
    // Smagorinsky SGS: sgs_n substeps of sgs_h seconds, the last sgs_h_last;
    // sgs_n = 0 when off
    int sgs_n;
    double sgs_h, sgs_h_last;
    int sgs_mode;                 // NIMBUS_SGS_*
    double sgs_c2d2;              // Cs^2 Delta^2
    double sgs_inv_pr, sgs_inv_sc; // 1 / Pr_t, 1 / Sc_t
    double sgs_nu_max, sgs_k_max;
    int sgs_wrap_x, sgs_wrap_y;   // periodic topology
    int sgs_open[4];              // west, east, south, north lateral faces open (radiative or zero-gradient)
    // explicit diffusion after the SGS: NIMBUS_DIFFUSE_* bits (0 off); when on,
    // the EOS projection and the sponges follow its commit instead of the
    // microphysics or SGS pass
    int dif_apply;
    double dif_kh, dif_kv;
    double dif_idx2, dif_idy2;  // 1 / (dx dx), 1 / (dy dy)
    int dif_wrap_x, dif_wrap_y;
    KesslerConst kessler;
    Bounds bounds;
};

// Launch geometry of one member: workgroups of tile_w x (256 / tile_w)
// columns (four waves of 64 lanes). Per-cell kernels visit the levels of a
// column tile consecutively within each of k_chunks vertical chunks
// (k_chunks = nz reproduces plane-by-plane order).
struct MemberGeom
{
    int tile_w, tile_h, tiles_x, tiles_y;
    int k_chunks;
    int xcd_remap;
    // per-cell work in runs of kBlock consecutive elements of one level's
    // padded [j][i] plane (`runs` per level) instead of column tiles at one level
    int linear, runs;
    // HE-VI solve: 16-byte lanes per level of a workgroup (solve_lanes) and
    // elements per 16 bytes (fixed by the storage type at creation)
    int solve_lanes, vec;
    // workgroups of the edge cells (close_edges), which the boundary closure spreads
    int edge_blocks;
};

// A low side that copies an open high side's face periodically needs that
// face before and after its closure, so the momentum update cannot close it.
__host__ __device__ inline bool bc_split(const StepParams& p)
{
    auto split = [](int lo, int hi) {
        return lo == NIMBUS_BC_PERIODIC && (hi == NIMBUS_BC_RADIATIVE || hi == NIMBUS_BC_ZERO_GRADIENT);
    };
    return split(p.bc_west, p.bc_east) || split(p.bc_south, p.bc_north);
}

struct MemberArgs
{
    DevGrid g;
    MemberGeom geo;
    DevFields f;
    StepParams p;
};

// Work shapes of a launch: what one map entry (one workgroup) covers.
enum WorkKind
{
    W_CELL = 0,    // one tile of columns at one level, or one run of a level (one cell per thread)
    W_DIAG = 1,    // one of kDiagBlocksPerMember reduction blocks
    W_SOLVE = 2,   // solve_lanes x 16 bytes consecutive columns of one row, whole columns (BatchView::solves)
    W_TILECELL = 3,  // one tile of columns at one level whatever the geometry (wide stencils)
    W_MOMENTUM = 4,  // a wind component of 256 edge cells (edge_blocks of them), then as W_CELL
    W_SHELL = 5,     // a wind component of 256 edge cells (edge_blocks of them), then 256 other columns
    W_KINDS = 6
};

// Column-solve form of a member (nimbus_hip_member_set_column_solve), at its
// creation PARTITIONED for FP64 members and for FP32 members of fewer than
// kSweepColumns columns, both up to kSegMaxNz levels. A name that is accepted,
// refused, reported and kept in snapshots; k_hevi_solve solves the columns of
// either form with the same operations.
constexpr int kSegMaxNz = 129;
constexpr int kSweepColumns = 32768;
constexpr bool hevi_partitioned_always(int elem, int nz) { return elem == 8 && nz <= kSegMaxNz; }
constexpr int hevi_default_seg(int elem, int nx, int ny, int nz)
{
    return nz <= kSegMaxNz && (elem == 8 || long(nx) * long(ny) < long(kSweepColumns)) ? 1 : 0;
}

// HE-VI solve: lanes of 16 bytes (vec elements) per level, so that a workgroup of
// one thread per lane holds a whole column of up to 1,024 levels (runtime grid
// check) in at most 1,024 threads. Workgroups of more than 8 waves go one to a
// CU: FP64 members of 129 to 160 levels take two lanes, of which several fit (ms
// per step with four lanes -> two: 128 x 128 x 129 1.61 -> 1.56, 160 x 160 x 140
// 2.95 -> 2.77, 48 x 48 x 140 0.42 -> 0.37). FP32 members there lose as often as
// they gain (48 x 48 x 140 6 % slower, 96 x 96 x 140 7 % faster), FP64 ones of 161
// to 192 levels lose 3 %.
constexpr int solve_lanes(int nz, int vec)
{
    return nz <= 256 && !(vec == 2 && nz > 128 && nz <= 160) ? 4 : nz <= 512 ? 2 : 1;
}

// Launch of the HE-VI solve for columns of up to nz levels, and how many of its
// workgroups a CU holds: 20 waves (the kernel's launch bound) and 160 KB of LDS.
struct SolveShape
{
    unsigned threads;
    std::size_t lds;
    int resident;
};
SolveShape solve_shape(int nz, int vec);

// Member subsets a launch can be restricted to.
enum MemberSubset
{
    S_ALL = 0,
    S_EXPLICIT = 1,
    S_HEVI = 2,
    S_SUBSETS = 3
};

struct BlockMap
{
    const int2* entries = nullptr;  // device: {member index, local work index}
    int blocks = 0;
};

// HE-VI members of a batch that one launch solves: columns of up to nz levels,
// all with the same lanes per level.
struct SolveGroup
{
    int nz = 0, lanes = 0;
    BlockMap map;
};

struct BatchView
{
    const MemberArgs* args = nullptr;  // device array
    int n = 0;
    int max_substeps = 0;
    int max_kessler_sub = 0;
    int any_sponge = 0;
    int max_sgs_n = 0;
    // parities that decide whether a copy-home kernel has work: some member
    // with an odd substep count (acoustic commit), an even microphysics
    // subcycle count (scalars home), an odd SGS substep count (SGS home)
    int any_odd_substeps = 0, any_even_kessler_sub = 0, any_odd_sgs_n = 0;
    int any_sponge_unfused = 0;  // a member with sponges and no SGS or diffusion pass to apply them in
    int any_diffusion = 0;       // a member with explicit diffusion
    int any_kessler_adaptive = 0; // a member whose microphysics subcycles follow its sedimentation limit
    int any_bc_split = 0;        // a member whose substeps are closed by k_close
    int max_nz = 0;
    std::vector<SolveGroup> solves;
    int elem = 4;
    BlockMap maps[S_SUBSETS][W_KINDS];
};

// Number of local work items of `kind` for one member.
int work_items(const MemberArgs& a, WorkKind kind);
void fill_geometry(MemberArgs& a, int tile_w, int k_chunks, int xcd_remap);

// Whole large step of every member of the batch.
template <class S>
void launch_large_step(Launcher& L, const BatchView& b);

// Individual phases (per-operation dispatch entry points).
template <class S>
void launch_slow_rk2(Launcher& L, const BatchView& b);
template <class S>
void launch_slow_tendencies(Launcher& L, const BatchView& b, void* du, void* dv, void* dw);
// Substep s of the acoustic loop (0-based): reads buffer s & 1, writes (s + 1) & 1;
// close: with its boundary closure, which radiates with the member's dts (the
// radiative faces start from the winds stored at substep 0).
template <class S>
void launch_acoustic_substep(Launcher& L, const BatchView& b, int s, bool accumulate, bool init_at_first, bool close);
// Boundary closure of the home buffers, without radiation.
template <class S>
void launch_boundaries(Launcher& L, const BatchView& b);
// Moves rho' from buffer 1 to buffer 0 for members whose last substep (n_done - 1) left it there.
template <class S>
void launch_commit(Launcher& L, const BatchView& b, int n_done);
template <class S>
void launch_transport(Launcher& L, const BatchView& b, int n_scalars, const int* pd, bool into_temp);
template <class S>
void launch_kessler_tendencies(Launcher& L, const BatchView& b, double dt, void* dth, void* dqv, void* dqc,
                               void* dqr);
template <class S>
void launch_diagnostics(Launcher& L, const BatchView& b);
// Elements [r0, r0 + nr) of the (j, k) planes of columns i0 .. i0 + ni - 1 of a
// host array [i][j][k], packed; nr is a whole plane where ni > 1.
struct HostPart
{
    int i0, ni, r0, nr;
};
// Device field (elements S, base profile subtracted) from or to such a part of
// a host array (elements H), at an address that the device can reach.
template <class S, class H>
void launch_turn(Launcher& L, const DevGrid& g, void* dev, void* host, const double* base_slot, bool to_host,
                 const HostPart& part);

constexpr int kDiagValues = 8;
constexpr int kDiagBlocksPerMember = 64;

}  // namespace nimbus
