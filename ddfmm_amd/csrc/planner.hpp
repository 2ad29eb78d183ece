// Host planner: builds the tree (Tree), fetches operators (Mlib) and flattens every
// stage of Wave3d::eval into descriptor tables (HostPlan) for the device.
#pragma once

#include <map>
#include <string>
#include <vector>

#include "host.hpp"
#include "plan.hpp"

namespace ddfmm {

struct PlanStats {
    int64_t npts = 0, nleaf = 0, nlf = 0, nhf_out = 0, nhf_in = 0;
    int64_t near_interactions = 0;      // sum over U/W/X-direct pairs of n_t * n_s (leaf kernel, point sources)
    int64_t near_mirrored = 0;          // near-field leaf pairs evaluated once for both directions
    int64_t leaf_op_interactions = 0;   // leaf kernel interactions with operator point sets (L2T, W via upeq)
    int64_t s2m_interactions = 0, x2chk_interactions = 0;
    int64_t v_pairs = 0, v_targets = 0, v_sources = 0;
    int64_t m2l_pairs = 0, m2l_groups = 0;
    double m2l_flops = 0, gemm_flops = 0;   // useful complex-GEMM flops (8*M*K*N) per RHS
    int64_t opmat_elems = 0, opmat_generated = 0;
    int nlevels_lf = 0, nlevels_hf = 0, max_hf_width = 0;
};

// A planned GEMM stage before it is cut into one launch per tile height: its groups, in
// order, and the largest tile height its tiling uses.
struct LogicalGemm {
    std::vector<int> groups;
    int mbmax = GEMM_MB;
    char name[24] = {0};
};

struct HostPlan {
    Params prm;
    int64_t N = 0;
    int P = 0, NL = 0;
    std::vector<int> perm;                 // sorted position -> input index
    std::vector<double> px, py, pz;        // leaf-sorted points then LF operator point sets
    std::vector<cpx> opmat;                // uploaded operator tables (prefix of the table)
    int64_t opmat_total = 0;               // uploaded + generated
    int64_t opmat_up = 0;                  // uploaded part alone
    std::vector<PackA> pack32, pack64;     // operator blocks packed at setup, per table
    int64_t pack32_total = 0, pack64_total = 0;   // with the slack behind them (GEMM_AHEAD)
    int64_t zeros = 0;                     // length of the GEMMs' block of zeros, behind the uploaded part
    bool stored = false;                   // FP64: the GEMMs read the table itself, nothing is packed
    std::vector<SetupWindow> windows;      // the generated part, in order
    int64_t window_elems = 0;              // the longest of them
    int pack_up[2] = {0, 0};               // packing jobs (FP64, FP32) from the uploaded part: the first ones
    std::vector<int> grid;                 // FFT grid index tables
    std::vector<double> genpts;            // kernel-generation point table (xyz rows)
    std::vector<KGen> kgen;
    std::vector<KTask> ktasks;
    std::vector<KSrc> ksrcs;
    std::vector<GGroup> groups;
    std::vector<double> group_flops;       // useful flops per RHS of each group
    std::vector<GTile> tiles;
    std::vector<int64_t> colB, colC, colA;
    std::vector<FftSrc> fsrc;
    std::vector<VTarget> vtrg;
    std::vector<VPair> vpair;
    std::vector<VChunk> vchunk;
    std::vector<int> vsrc;                  // chunk source unions (spectrum indices)
    std::vector<int> vpk;                   // packed pairs per target, padded to multiples of 8
    std::vector<RTarget> rtrg;
    std::vector<Stage> stages;
    std::vector<Stage> setup_stages;       // FP64 GEMMs on the operator table, window by window
    int setup_t0 = 0, setup_t1 = 0;        // their tiles
    std::vector<LogicalGemm> lgemm;        // logical GEMM stages of `stages` (Stage::lstage)
    int64_t bufsize[BUF_COUNT] = {0};      // elements per rhs
    PlanStats stats;
    std::string dump;                      // canonical text of the lists (debug/parity)

    int64_t vector_bytes() const { return prm.xlat > 0 ? 8 : 16; }    // of a work buffer's element
    int64_t rhs_bytes() const {            // work buffers and staging of one right-hand side
        int64_t n = 0;
        for (int64_t b : bufsize) n += b;
        return N * 16 + n * vector_bytes();
    }
    // what setup holds besides the tables it leaves and the window
    int64_t setup_bytes() const {
        return (int64_t)(genpts.size() * sizeof(double) + kgen.size() * sizeof(KGen) +
                         (stored ? 0 : pack32.size() + pack64.size()) * sizeof(PackA));
    }
    // GGroup::transA of a stage's groups: 2 or 3 packed, 0 as stored (in either order)
    int gemm_form(const Stage& s) const {
        const bool translation = s.prec == PREC_TRANSLATION;
        return stored || (translation && prm.xlat == 2) ? 0 : translation && prm.xlat == 1 ? 2 : 3;
    }
};

void build_plan(const Params& prm, const double* pos, int64_t N, const Mlib& mlib,
                HostPlan& plan, bool want_dump);

// Device bytes of a set-up context: `fixed` for the point, operator and descriptor tables
// (kept for the context's life), `per_rhs` for the work buffers and the staging of one
// right-hand side, `setup` for what lives during setup only (under a budget freed before the
// work buffers are allocated): the window of the operator table's generated part that is
// being made, the generator tables and the packing jobs.
struct PlanBytes {
    int64_t fixed = 0, per_rhs = 0, setup = 0;
};
PlanBytes plan_bytes(const HostPlan& plan);

// Throws unless every descriptor's range lies inside the buffer or table it indexes
// (build_plan ends with it).
void validate_plan(const HostPlan& plan);

// Algorithmic work per RHS of a stage (Stage::work) and, for GEMM stages, the MFMA flops
// the kernel executes under its tiling (Stage::exec).
void stage_work(const HostPlan& plan, Stage& s);

// Rebuild the tiles of every logical GEMM stage with at most mbmax[l] row blocks of 16 per
// tile (1..GEMM_MB; a group's rows spread evenly over ceil(blocks / mbmax) tiles) and the
// GEMM launches of `stages` (one per tile height), after setup: the setup-time GEMMs'
// tiles are dropped.  Other stages keep their order.
void retile(HostPlan& plan, const std::vector<int>& mbmax);

}  // namespace ddfmm
