// sgk_internal.h - host-side engine context and the kernel launchers of each translation unit.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "sgk.h"
#include "sgk_adjoint.h"
#include "sgk_batch.h"
#include "sgk_params.h"
#include "sgk_xfer.h"

namespace sgk {

// Buckets per block of the two-pass counting-sort scan (k_ord_blocksum / k_ord_scan); the block-total
// arrays hold one int per kOrdChunk buckets.
constexpr int kOrdChunk = 1024;

struct GraphEntry {
    hipGraphExec_t exec = nullptr;
    unsigned long long uses = 0;
};

struct KernelStat {
    int launches = 0;
    double ms = 0;
};

}  // namespace sgk

struct sgk_ctx {
    SimParams sp;
    sgk_config cfg;
    sgk::DevParams dp;
    bool mixed = false;
    int device = 0;
    hipStream_t stream = nullptr;

    // state arrays (positions AoS x,y,z,E; velocity and acceleration SoA, storage precision R)
    void *pos = nullptr;   // float4 or double4 [nMol]
    void *posAlt = nullptr;  // the same: where a force pass with the fused drift writes the next positions
    void *vel = nullptr;   // R [3*nMol]
    void *acc = nullptr;   // R [3*nMol] (FP64 in the mixed form)
    float *rho = nullptr, *embF = nullptr, *embDF = nullptr, *fric = nullptr;  // [nMolMe]
    // cells (two buffers, see the rebuild protocol in sgk_nebr.hip)
    int *cellOf[2] = {nullptr, nullptr};
    int *cnt[2] = {nullptr, nullptr};
    int *slots[2] = {nullptr, nullptr};
    int *slotOf = nullptr;
    float4 *cellPos = nullptr;
    // neighbour structures
    int *nlM = nullptr, *nnM = nullptr;                 // metal: row-major [nMolMe*nlCap]
    unsigned int *lj = nullptr, *cl = nullptr;          // carbon: column-major packed (idx<<8|pos)
    int *nlj = nullptr, *ncl = nullptr;
    uint4 *bondC = nullptr, *bondA = nullptr;          // carbon: per-step near lists (k_rho)
    int *fullNN = nullptr, *fullNBL = nullptr;          // reference layout (keep_full_nl)
    // order in which nl_scheme 3 builds the carbon lists (carbons by cell, then metal atoms) and the
    // counting-sort scratch that makes it (sgk_nebr.hip)
    int *nlOrder = nullptr, *ordCnt = nullptr, *ordKey = nullptr, *ordSlot = nullptr, *ordBlock = nullptr;
    bool orderValid = false;
    int orderAge = 0;                                   // steps run since the order was built
    // reductions and run state
    void *partials = nullptr;
    void *partVmax = nullptr;                           // v^2 maximum of every force-pass workgroup
    void *partialsAlt = nullptr, *partVmaxAlt = nullptr;  // swapped with state, below
    sgk::DevState *state = nullptr;
    sgk::DevState *stateAlt = nullptr;                  // swapped with state inside a chunk of steps, never across one
    sgk_record *records = nullptr;
    unsigned int *hist = nullptr;
    sgk::DevState *hostState = nullptr;                 // pinned mirror
    sgk::HostStage stage;                               // state transfer, grown on demand
    // launch geometry
    int block = 256, metalLanes = 8, carbonLanes = 1, nbM = 0, nbC = 0, nbRho = 0, nbProps = 0;
    int part2Off = 0;                                   // chunk totals of the step reduction (in partials)
    long long bytes = 0;
    bool haveList = false;
    bool haveCells = false;                             // sgk_bin ran on the current positions
    int hostStep = 0;                                   // host copy of the step counter
    double lastRunMs = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::map<std::string, sgk::GraphEntry> graphs;
    bool profiling = false;
    std::map<std::string, sgk::KernelStat> stats;
    std::string err;
    sgk::Adjoint *adj = nullptr;                        // adjoint storage (sgk_adjoint_*), on demand
    sgk::DiffusionArgs diff = {};                       // device diffusion (sgk_diffusion_enable), on demand
    void *diffMem = nullptr;
    // complete-range RDF (cfg.rdf_complete): metal atoms sorted by the RDF grid at each sample
    sgk::RdfGrid rdfGrid = {};
    int *rdfCnt = nullptr, *rdfKey = nullptr, *rdfSlot = nullptr, *rdfBlock = nullptr;
    float4 *rdfPos = nullptr;
};

// A batch of replicas advanced together (sgk_batch_*): shared arrays, one range per replica.
namespace sgk {
// Lanes per metal atom of the cell-ordered list build (each takes two of every 2G candidates; 8
// measured no faster on the batch and 1.5 % slower on the 1.1 M-atom system).
constexpr int kNlMetalLanes = 4;
// Atoms per workgroup of the nine-lane list build (four waves of seven atoms), and the largest system
// (or batch, atoms of all replicas) that uses it.  The nine-lane build is shorter in latency, the
// one-lane build in instructions; whole steps at 900-1,000 K, one-lane / nine-lane (us): 1,161 atoms
// 39.3 / 34.6, 44,353 49.8 / 41.0, 129,120 53.1 / 48.0, 275,880 85.7 / 84.8, 440,000 107.7 / 114.9,
// 1.1 M 224 / 248; batches of 373,577 atoms 112.9 / 113.0, of 448,542 125.0 / 127.4.
// A metal atom has four lanes otherwise, and a column of its cells up to 72 candidates: it pays for nine lanes only beside
// carbons, whose one lane under a cluster is the longest chain of the launch.  A rebuild on thermal
// positions, four lanes / nine: bulk metal 10,976 atoms 50.6 / 36.8, 19,652 52.5 / 46.7, 32,000 49.8 / 57.6, 108,000
// 99.4 / 145, 256,000 169 / 294; clusters on a sheet, 30,000 + 3,520 C 86.2 / 52.4, 60,000 + 53,760 C 105 / 84.3,
// 100,000 + 30,720 C 128 / 111, 150,000 + 30,720 C 147 / 150, 200,000 + 53,760 C 184 / 199.
constexpr int kNineAtoms = 4 * 7;
constexpr int kNlNineAtoms = 1 << 18, kNlNineMetal = 1 << 17, kNlNineBulk = 28 << 10;
inline bool nl_nine(long long nC, long long nMe) {
    return nC + nMe <= kNlNineAtoms && nMe <= (nC > 0 ? kNlNineMetal : kNlNineBulk);
}
// A system, or a batch in all, of up to so many carbons takes four lanes per carbon in the density and
// force passes: there one lane's chain, not the chip's throughput, sets the time.  The results are the
// same bits either way.  Whole step with one lane / four (us), FP64 pairs unless said: 1,161 atoms
// 27.3 / 21.1, 18,896 29.5 / 25.4, 50,208 34.6 / 33.9, 60,448 34.9 / 36.0; FP32 17,196 24.9 / 21.1, 33,768
// 27.3 / 23.5; 14 replicas of 31,901 together 38.1 / 35.2, 64 of 413,000 107 / 126.
constexpr int kQuadCarbons = 49152;
inline int carbon_lanes(long long nC) { return nC <= kQuadCarbons ? 4 : 1; }
// Carbon workgroups that store a partial: one per 256 carbons, in four parts with four lanes.
inline int carbon_blocks(long long nC, int lanes) { return (int)((nC + 255) / 256) * lanes; }
// Reference-stencil RDF.
constexpr int kRdfAtoms = 8;          // atoms a workgroup takes at once
// Workgroups per launch at most: each merges its bins into one histogram, and fewer leave too few waves in
// flight.  A sample by one lane per atom / 512 workgroups of a run of atoms each / 512 taking groups in turn / 1,024 /
// 2,048 so (us, mixed, then FP32): clusters of 30,000 257 / 82 / 77 / 73 / 73, 238 / 72 / 68 / 61 / 71; 100,000
// 308 / 242 / 218 / 198 / 186, 282 / 190 / 176 / 130 / 122; bulk metal of 256,000 683 / 704 / 612 / 561 / 563,
// 514 / 592 / 510 / 367 / 339; of 864,000 1,590 / 2,087 / 1,822 / 1,573 / 1,588, 1,230 / 1,803 / 1,468 / 1,012 / 1,005.
constexpr int kRdfBlocks = 1024;
inline int rdf_chunk(long long nMe) {  // atoms per workgroup (at least one group)
    const long long groups = (nMe + kRdfAtoms - 1) / kRdfAtoms;
    return kRdfAtoms * (int)std::max<long long>(1, (groups + kRdfBlocks - 1) / kRdfBlocks);
}
}

// Force-pass workgroups of nMe metal atoms at G lanes each.  With the density or force pass
// remapped to XCDs (xcd_map bit 1 or 2) the count is padded to a multiple of 8, so that the carbon
// range starts on XCD 0; without, the padding workgroups would only idle.
inline int metal_blocks(long long nMe, int G, int xcdMap) {
    const long long nb = (nMe * G + 255) / 256;
    return (int)((xcdMap & 6) ? (nb + 7) / 8 * 8 : nb);
}

// Most partials of a step that k_lf1_next closes (it takes no chunk totals).  Each of its
// workgroups reads them all, and that still costs less than the launches it replaces: whole step
// without / with it (us), sheared FP32 9,417 atoms 24.8 / 21.5, 47,776 36.0 / 32.6, 119,200 43.7 / 42.0,
// mixed 119,200 53.8 / 53.2; deposition 17,196 24.1 / 19.0, 205,100 67.9 / 53.0.
constexpr int kCloseLf1Parts = sgk::kFoldParts;
// Most replicas of a batch with synchronised rebuilds whose steps are folded: every workgroup of
// kb_bin_next goes through all of them.  Whole step with closing launches / folded (us): 500 replicas of 525 atoms
// (FP32) 64.3 / 59.9, 1,000 99.6 / 93.5, 1,500 132.1 / 130.9, 2,000 168.8 / 176.9, 4,000 363 / 454; 1,000 of 1,161
// (mixed) 356.9 / 354.3, 2,000 740 / 766.
constexpr int kFoldSync = 1024;
// The force pass's partials of a step.
inline sgk::PartMap part_map(const sgk_ctx *c) { return {c->nbM, c->nbM + c->nbC, c->carbonLanes == 4}; }

struct sgk_batch {
    int nrep = 0;
    std::vector<SimParams> sp;
    sgk_config cfg;
    bool mixed = false;
    int device = 0;
    hipStream_t stream = nullptr;
    int metalLanes = 4;                 // the common lanes per metal atom (0 when replicas differ)
    std::vector<int> repLanes;          // lanes per metal atom of each replica
    // density and force passes: one launch per distinct lane count, its blocks at forceTab[grpOff[g]]
    static constexpr int kLaneKinds = 5;  // 1, 2, 4, 8, 16
    int grpOff[kLaneKinds] = {}, grpN[kLaneKinds] = {};
    std::vector<sgk::BatchRep> reps;  // host copy of the replica table
    sgk::BatchRep *dReps = nullptr;
    int2 *atomTab = nullptr, *forceTab = nullptr, *metalTab = nullptr, *nlTab = nullptr, *rdfTab = nullptr;
    int nAtomBlocks = 0, nForceBlocks = 0, nMetalBlocks = 0, nNlBlocks = 0, nRdfBlocks = 0;
    bool nlNine = false;  // nl_scheme 3 with nine lanes per atom (nlTab counts its workgroups)
    // cell-ordered list build (nl_scheme 3): the order of every replica from one counting sort
    int *order = nullptr, *ordCnt = nullptr, *ordKey = nullptr, *ordSlot = nullptr, *ordBlock = nullptr;
    long long nOrdBuckets = 0;
    bool orderValid = false;
    int orderAge = 0;
    long long nAtoms = 0, nMetal = 0, nCarbon = 0, nCells = 0;
    void *pos = nullptr, *vel = nullptr, *acc = nullptr;
    void *posAlt = nullptr;  // where a force pass with the fused drift writes the next positions
    float *rho = nullptr, *embF = nullptr, *embDF = nullptr, *fric = nullptr;
    int *cellOf[2] = {nullptr, nullptr}, *cnt[2] = {nullptr, nullptr}, *slots[2] = {nullptr, nullptr};
    int *slotOf = nullptr;
    float4 *cellPos = nullptr;
    int *nlM = nullptr, *nnM = nullptr, *nlj = nullptr, *ncl = nullptr;
    unsigned int *lj = nullptr, *cl = nullptr;
    uint4 *bondC = nullptr, *bondA = nullptr;
    void *partials = nullptr, *partialsAlt = nullptr;  // the Alt ones swapped inside a chunk of steps, as in sgk_ctx
    sgk::DevState *state = nullptr, *stateAlt = nullptr;
    unsigned long long *vmax = nullptr, *vmaxAlt = nullptr;
    bool canFold = false;                // every replica's partials can be closed by the next step's kernels
    sgk_record *records = nullptr;
    unsigned int *hist = nullptr;
    sgk::DevState *hostState = nullptr;  // pinned mirror, nrep entries
    sgk::HostStage stage;                // state transfer, grown on demand
    long long bytes = 0;
    int hostStep = 0;
    double lastRunMs = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::map<std::string, sgk::GraphEntry> graphs;
    std::string err;
    std::vector<void *> allocs;

    sgk::BatchArgs args() const {
        sgk::BatchArgs a;
        a.reps = dReps;
        a.atomTab = atomTab;
        a.forceTab = forceTab;
        a.metalTab = metalTab;
        a.nlTab = nlTab;
        a.rdfTab = rdfTab;
        a.order = orderValid ? order : nullptr;
        a.pos = pos;
        a.posOut = nullptr;
        a.vel = vel;
        a.acc = acc;
        a.rho = rho;
        a.embF = embF;
        a.embDF = embDF;
        a.fric = fric;
        for (int k = 0; k < 2; ++k) {
            a.cellOf[k] = cellOf[k];
            a.cnt[k] = cnt[k];
            a.slots[k] = slots[k];
        }
        a.slotOf = slotOf;
        a.cellPos = cellPos;
        a.nlM = nlM;
        a.nnM = nnM;
        a.nlj = nlj;
        a.ncl = ncl;
        a.lj = lj;
        a.cl = cl;
        a.bondC = bondC;
        a.bondA = bondA;
        a.partials = partials;
        a.partialsOld = partialsAlt;
        a.state = state;
        a.stateOld = stateAlt;
        a.vmax = vmax;
        a.vmaxOld = vmaxAlt;
        a.records = records;
        a.recCap = cfg.records_capacity;
        a.hist = hist;
        return a;
    }
};

namespace sgk {

// Device parameters of one system (sgk_api.hip).
void make_dev_params(const SimParams &s, const sgk_config &cfg, DevParams &p);
// Validates the parameters and the configuration (defaults filled in) and sets c->sp, cfg, mixed, dp
// and the launch geometry (lanes per metal atom, block counts, partials layout); allocates nothing.
// Returns SGK_OK or an error code with the reason in err.
int prepare_ctx(const SimParams *sp, const sgk_config *cfg, sgk_ctx *c, std::string &err);

// sgk_nebr.hip
void launch_bin(sgk_ctx *c, bool force);
// The previous step's closing decision (its state in c->stateAlt), then the binning of a rebuild step.
void launch_bin_next(sgk_ctx *c);
void launch_batch_sortcells(sgk_batch *b);
void launch_batch_nl(sgk_batch *b);
void build_batch_nl_order(sgk_batch *b);
void launch_batch_rdf(sgk_batch *b);
void launch_sortcells(sgk_ctx *c, bool force);
void launch_nl(sgk_ctx *c, bool force);
void build_nl_order(sgk_ctx *c);
constexpr int kNlOrderSteps = 100;  // age (steps) at which sgk_run rebuilds the nl_scheme 3 list-build order
void launch_commit_rebuild(sgk_ctx *c);
void launch_rdf(sgk_ctx *c);
RdfGrid rdf_grid(const DevParams &p, int S);  // complete-range RDF grid, cells range/S (ncell 0: range too large)
// sgk_force.hip
void launch_rho(sgk_ctx *c);
void launch_batch_rho(sgk_batch *b);
int batch_lane_index(int G);  // position of G in the lane kinds 1, 2, 4, 8, 16
// closePrev: the first workgroups close the previous step; fold: the next step closes this one (it takes the maxima).
void launch_batch_force(sgk_batch *b, bool prekick = false, void *posOut = nullptr, bool closePrev = false,
                        bool fold = false);
void launch_batch_force_eval(sgk_batch *b);  // forces and energies only: velocities untouched
// prekick: the force pass also applies the next step's first half-kick (the caller guarantees that
// nothing touches velocities or accelerations before that step's launch_lf1(kicked = true)).
// posOut (with prekick): also drift the positions of the next step into posOut (sgk_force.hip).
// closePrev: one more workgroup closes the previous step (its state and partials in the Alt buffers).
void launch_force(sgk_ctx *c, bool integrate, bool finalize, bool prekick = false, void *posOut = nullptr,
                  bool closePrev = false);
// sgk_step.hip
void launch_lf1(sgk_ctx *c, bool bin, bool kicked = false);
void launch_insert(sgk_ctx *c);
void launch_lf1_next(sgk_ctx *c, bool shear);  // with the closing of a folded step (regime 1: and the insertion)
// drifted: the previous force pass drifted the positions (posOut), so only the binning is left.
void launch_batch_lf1(sgk_batch *b, bool kicked = false, bool drifted = false, bool folded = false);
void launch_batch_finalize(sgk_batch *b);
void launch_batch_thermostat(sgk_batch *b);
void launch_batch_shear(sgk_batch *b);
void launch_batch_reset_records(sgk_batch *b);
void launch_lf2(sgk_ctx *c);
void launch_props(sgk_ctx *c);
void launch_finalize(sgk_ctx *c, int mode);          // 0 step, 1 evaluate only
void launch_reduce_chunks(sgk_ctx *c);
void launch_thermostat(sgk_ctx *c, int stepOverride, double vvOverride, int useOverride);
void launch_shear(sgk_ctx *c);
void launch_reset_records(sgk_ctx *c);
void launch_diffuse(sgk_ctx *c);
void launch_diffuse_reset(sgk_ctx *c);

// sgk_api.hip: error reporting, device flags, the step-kernel flags of a run and the device loop.
int set_error(sgk_ctx *c, int code, const std::string &msg);
int check_device_flags(sgk_ctx *c);
// One character per step, 'a' + bits: 1 thermostat, 2 shear, 4 RDF, 8 adhesion energy recorded,
// 16 diffusion sample.
std::string step_flag_string(sgk_ctx *c, int step0, int nsteps, int rdfEvery, bool observe);
// Where the positions of the steps are kept: after step k they lie at slot(k), and stay there.  after(k) runs
// when step k's force pass is enqueued, before its thermostat.
struct StepTrace {
    char *pos = nullptr;
    size_t stride = 0;
    std::function<int(size_t)> after;
    int rc = 0;
    char *slot(size_t k) const { return pos + stride * k; }
};
// Enqueues the steps of the flags; with a trace, c->pos ends on its last slot.
void enqueue_steps(sgk_ctx *c, const std::string &flags, StepTrace *trace = nullptr);
// sgk_run with, if adh is not null, the adhesion energy of every step copied to adh[nsteps].
int run_steps(sgk_ctx *c, int nsteps, int rdfEvery, sgk_record *records, double *adh);
// Destroy the cached step graphs (their launches carry grids, parameters and buffer addresses).
void drop_graphs(sgk_ctx *c);

// Per-kernel timing hook used when profiling is on (sgk_api.hip).
void profile_begin(sgk_ctx *c);
void profile_end(sgk_ctx *c, const char *name);

// Partial-record size for the context precision.
size_t partial_bytes(const sgk_ctx *c);
size_t partial_bytes_for(bool mixed);

}  // namespace sgk
