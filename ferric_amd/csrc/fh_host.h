// Host-side state and helpers shared by the C ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <utility>
#include <vector>

#include "../../include/ferric_hip.h"
#include "fh_kernels.h"

namespace fh {

enum SlotId {
    kSlotStage = 0,  // FP64 staging copy of a host b_ov
    kSlotOp0,        // packed operand (or BF16 hi)
    kSlotOp1,        // BF16 lo
    kSlotScale,      // FP8 scales
    kSlotEps,        // eps_occ | eps_vir
    kSlotItems,      // per-item partial sums
    kSlotRows,       // per-row partial sums
    kSlotResult,     // energies + row values
    kSlotScalar,     // small scalars (absmax)
    kSlotGamma,      // adjoint: FP64 gamma staging for host calls
    kSlotT,          // adjoint: per-row T~ block, or the whole amplitude matrix
    kSlotDeps,       // adjoint: dE/deps partials
    kSlotBatch,      // batched: descriptors and work list
    kSlotBatchOut,   // batched: per-domain partials
    kSlotAcc,        // adjoint: compensated dE/deps sums of the rows so far
    kSlotDiag,       // BF16: lo^2 row sums
    kSlotStage2,     // adjoint: Q-major padded copy of B
    kSlotU,          // adjoint: b-major T~ blocks of one row, or B by Q
    kSlotSplit,      // adjoint: split-K partial tiles of phase B
    kSlotRed,        // adjoint: reduction partials of a batch of rows
    kSlotDressX,     // dressing: (Q|nu i) half-transformed rows
    kSlotDressY,     // dressing: undressed MO rows (Q|ia)
    kSlotB2Split,    // INT8X4 adjoint: BF16 hi and lo of the Q-major copy of B
    kSlotTSplit,     // INT8X4 adjoint: BF16 hi and lo of a row group's T~ slabs S and St
    kSlotG32,        // INT8X4 adjoint: FP32 gamma over the padded index space
    kSlotPairs,      // pair energies: (e_os, e_ss) per unique pair
    kSlotPnoWork,    // PNO: five nvir x nvir matrices and three vectors per batched pair
    kSlotPnoMeta,    // PNO: pair list, per-pair results, masks, GEMM pointer arrays
    kSlotFitWork,    // domain fits: eliminated rows of [V_DD | A_i | A_j] per batched pair
    kSlotFitMeta,    // domain fits: aux bits per occupied, pairs, domain lists, pivot info
    kSlotGPairs,     // energies from explicit (ia|jb) blocks: the pair list
    kSlotRexpB,      // INT8X4 opposite spin: row exponents of the beta rows
    kSlotDensAmp,    // MP2 densities: amplitude blocks of every ordered occupied pair
    kSlotDensPart,   // MP2 densities: split-K partial tiles
    kSlotDensOut,    // MP2 densities: P_vv (padded) then P_oo
    kSlotResidue,    // residue arithmetic: the workgroups' residue planes
    kSlotRange,      // residue arithmetic: column maxima and sums of B (no entry stages an
                     // input here, as some do in kSlotStage and kSlotStage2)
    kNumSlots
};

struct Slot {
    void *ptr = nullptr;
    size_t bytes = 0;
    bool spare = false;  // grown for a route that has another behind it (reserve)
};

struct Pending {
    uint64_t h2d_bytes = 0, d2h_bytes = 0, kernel_launches = 0;
    uint64_t slots = 0;  // bit k: slot k belongs to this call
};
static_assert(kNumSlots <= 64, "Pending::slots is one word");

struct GraphCache;  // batched.hip

struct State {
    std::mutex mu;
    bool initialised = false;
    int device = 0;
    size_t pool_limit = 0;
    bool pool_limit_explicit = false;
    Slot slots[kNumSlots];
    fh_stats stats{};
    Pending pending;
    GraphCache *graphs = nullptr;
    void *blas = nullptr;  // rocBLAS handle of the device, made on first use (blas_handle)
    // Phase timing (FERRIC_TIMING): events on the call's stream.
    int timing = -1;  // -1: not yet read from the environment
    int wall_khz = -1;  // device wall-clock rate (kHz); -1: not yet queried
    int cus = 0;        // compute units; 0: not yet queried
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    fh_timing last_timing{};
    // Fixed arena (fh_rimp2_energy_dev_noalloc): while set, reserve() carves
    // the requested slots out of it in request order and never allocates.
    char *arena = nullptr;
    size_t arena_bytes = 0, arena_used = 0;
    // Pinned host memory of kHostDoubles: results written by the reductions and
    // orbital energies read by the packer, instead of pageable copies. Calls hold `mu`
    // and end with a stream sync, so it serves one at a time; fh_release_workspace
    // frees it.
    double *host = nullptr;
    // Orbital energies on their way to the device where `host` does not take them: the
    // copy reads them until the call's stream sync.
    std::vector<double> eps_up;
    size_t held_bytes() const;
};

// Phase markers: record(k) for k = 0 (start), 1 (after pack), 2 (after the
// contraction), 3 (after the reductions); finish() after the stream sync.
bool timing_on(State &s);
// Wall-clock ticks per Q panel for the INT8X4 kernels' panel rotation (0: off)
// for a problem of npanels 64-deep Q panels and ntp tile pairs per occupied pair.
int i8_q_rot_ticks(State &s, int npanels, int ntp);
void mark(State &s, int k, hipStream_t st);
void finish_timing(State &s, uint64_t items, int tile);

struct EnergyPlan {
    int tile = 128;
    int nvir_pad = 16;
    int naux_pad = 128;
    int ntile = 1;
    int ntp = 1;
    int64_t nitems = 0;
    int group = 1;  // residue arithmetic: occupied orbitals side by side in a tile
};

State &state();
fh_status fail(fh_status st, const char *fmt, ...);
void clear_error();
fh_status ensure_device(State &s);
// spare: for a route that has another behind it. What it grows is given back as soon as a
// later call, or that other route, does not fit beside it, so that no call is refused for
// the sake of a faster route's workspace.
fh_status reserve(State &s, const std::vector<std::pair<int, size_t>> &req, bool spare = false);
// A route with another behind it: undo() after its FH_POOL_FULL, before the other is tried.
// The failure is not counted, and the slots it reserved no longer belong to the call.
struct Attempt {
    State &s;
    uint64_t full, slots;
    explicit Attempt(State &st)
        : s(st), full(st.stats.fail_pool_full), slots(st.pending.slots) {}
    void undo() const {
        s.stats.fail_pool_full = full;
        s.pending.slots = slots;
        clear_error();
    }
};
void release_all(State &s);
fh_status hip_check(hipError_t e, const char *what);
fh_status check_shapes(size_t naux, size_t nocc, size_t nvir, size_t n_eps, size_t first_occ,
                       size_t nocc_total, bool *empty);
fh_status check_kappa(double kappa, bool *has);
// wide: also the flag of the residue range test, the second word of kSlotScalar.
fh_status range_check(State &s, const void *b, bool in_f32, size_t n, size_t depth,
                      hipStream_t stream, bool *wide = nullptr);
EnergyPlan plan_energy(size_t nocc, size_t nvir, size_t naux, Prec prec);
// FERRIC_HIP_TILE's tile side, or 0 when it is unset.
int forced_tile();
// FERRIC_HIP_TILE=256: residue arithmetic wherever it can run.
bool forced_residue();
// Tile side of n batched domains: FERRIC_HIP_TILE's if set, else the first
// tile-table entry whose bounds hold the domain, else 0 (one environment
// read, one lock).
void tuned_tiles(Prec prec, size_t n, const size_t *nvir, const size_t *naux, int *out);
size_t packed_elem_bytes(Prec p);
// The device's rocBLAS handle (created on first use, atomics off so that its
// GEMMs are deterministic), bound to stream.
fh_status blas_handle(State &s, hipStream_t stream, void **handle);
// Bytes of one packed operand array of plan pl (INT8X4 adds TILE spare rows).
size_t packed_op_bytes(const EnergyPlan &pl, size_t nocc, Prec prec);
// neg_dev (naux_neg rows, same layout and dtype as b_dev) makes the kernel
// signed: K = B^T B - N^T N (FP64 / FP32 only).
fh_status energy_core(State &s, const void *b_dev, fh_dtype b_dtype, size_t naux, size_t nocc,
                      size_t nvir, const double *eps, size_t first_occ, size_t nocc_total,
                      double kappa, Prec prec, hipStream_t stream, fh_spin_components *out,
                      double *row_partials, const EnergyPlan *forced,
                      const void *neg_dev = nullptr, size_t naux_neg = 0,
                      const AmpOut *amp_out = nullptr, int *ntp_used = nullptr,
                      bool as_noalloc = false);
constexpr size_t kHostDoubles = 8192;
// The pinned buffer, or null: more than it holds, the fixed arena (no allocation), or none
// to be had.
double *host_buffer(State &s, size_t doubles);
int compute_units(State &s);  // of the device, asked once; at least 1
// Residue arithmetic (residue.hip). Tile sides and paddings of a shape, where it may
// run at all (aux count, forced tiles, fixed arena); whether an energy of this
// shape is faster so, and its plan; and the workspace of a launch.
bool residue_tiles(State &s, size_t nvir, size_t naux, EnergyPlan *pl);
// Whether it is faster: FLOP and 64 x 64 items of the padded problem on the matrix kernel.
bool residue_pays(const ResidueShape &p, size_t nocc, int nvir_pad, size_t nocc_b, int nvir_pad_b,
                  size_t naux);
struct ResidueSpace {
    ResidueArgs args;    // prec, np, beta, op, rexp, nitems, blocks, scratch, queue, order
    ResidueOrder order;  // words, queue, order
    ResidueRange range;
    int8_t *op = nullptr;
    int *rexp = nullptr;
    int *wide = nullptr;
};
// nov: columns of B, rows: packed rows, norb: occupied orbitals (both sides' together), nvir:
// the larger side's.
fh_status reserve_residue(State &s, Prec prec, int64_t nitems, int products, size_t nov,
                          size_t rows, size_t norb, size_t nvir, int naux_pad,
                          std::vector<std::pair<int, size_t>> more, ResidueSpace *out);
// Copies the device result (energies, then nocc rows' values, then, if asked for, the residue
// kernel's flag) back and waits for it.
fh_status fetch_result(State &s, const double *dev, size_t nocc, hipStream_t stream,
                       fh_spin_components *out, double *row_partials, bool *wide = nullptr);
bool plan_residue(State &s, size_t nocc, size_t nvir, size_t naux, Prec prec, EnergyPlan *pl);
void commit(State &s, Prec prec, bool adjoint, bool batched);
bool to_prec(int p, Prec *out);
void release_graphs(State &s);

}  // namespace fh
