// cmf_block.hpp -- several substeps of a model in one launch (cmf_block.hip):
// the partition of the river network into blocks and its launch.
#pragma once
#include "cmf_device.hpp"
#include <vector>

namespace cmf {

// Partition of the network (host): nblk blocks of T local cells. A block owns
// some cells (whole basins, and connected parts of basins larger than a block)
// and holds beside them the cells its owned ones depend on over kmax substeps.
struct BlockPlan {
    int T = 0, kmax = 0, nblk = 0;
    bool closed = false;                       // no block holds a cell of another: any number of substeps
    std::vector<int32_t> cell;                 // [nblk*T] device cell of each local cell, -1 idle
    std::vector<uint32_t> topo;                // [2][nblk*T], the fields below
    std::vector<int32_t> upx_ptr;              // [nblk*T] start of the list in upx of cells with more than two
    std::vector<uint16_t> upx;
    std::vector<int32_t> ndam;                 // [nblk] dam cells | kinematic cells << 16
    std::vector<int32_t> dom;                  // [nblk] domain of the block's cells
    // bifurcation paths (empty without): thread of a block -> path and level of its wavefront, packed
    // with the ends and codes; path slots of a cell, the third on in ppx
    std::vector<int32_t> path;                 // [nblk*T] path or -1
    std::vector<uint32_t> pword, pends;        // [nblk*T] PATH_* fields; [nblk*blk_paths(T)] ends of a slot
    std::vector<uint32_t> pcell;               // [nblk*T] first two slots (8 bits each), paths out and in (8 each)
    std::vector<int32_t> ppx_ptr;              // [nblk*T]
    std::vector<uint16_t> ppx;
};
// dam cell (any), levee cell, reads its upstream cells' flows, dam cell on the kinematic wave
enum : uint8_t { BLK_DAM = 1, BLK_LEV = 2, BLK_DAMUP = 4, BLK_KINE = 8 };
// The network in device cell order: downstream cells, upstream lists, BLK_* flags
// (NULL: none), domains (ascending, NULL: one; a block's cells share theirs), and the
// bifurcation paths with both ends in the network (lists of those out of and into a
// cell; npth = 0: none).
struct BlockNet {
    int n;
    const int32_t *next, *up_ptr, *up_idx;
    const uint8_t* special;
    const int32_t* domain;
    int npth, npthlev;
    const int32_t *pth_up, *pth_down, *out_ptr, *out_idx, *in_ptr, *in_idx;
};
// False when the network cannot be cut into such blocks (a cell with too many
// upstream cells, or whose surroundings alone overfill a block), not into max_blocks of
// them, or, with closed_only, not into blocks of whole basins; as soon as that is known.
bool build_block_plan(const BlockNet& net, int T, int kmax, bool closed_only, int64_t max_blocks, BlockPlan& out);

// Order of the cells of a block: dam cells from 0, kinematic cells (above a dam)
// from BLK_KINE_AT, so that the two rare flow rules are computed by different
// wavefronts; levee cells take the lowest places left. Their extra state has LDS
// slots for so many of each.
constexpr int BLK_KINE_AT = 64;
constexpr int blk_dams(int T) { return T / 32; }
constexpr int blk_kines(int T) { return 3 * T / 32; }
constexpr int blk_special(int T) { return 3 * T / 8; }
constexpr int blk_paths(int T) { return T / 4; }            // blocks along paths have 512 cells at most

// The levels of a path are computed by neighbouring lanes, whole paths in a wavefront,
// from the last one of the block down (the ring's, which has least to do otherwise).
// Word of such a thread: level (6 bits), slot (8), code (6); ends of a slot: local cells
// (10 bits each), flags set by the kernel
constexpr int PATH_SLOT = 6, PATH_CODE = 14;
constexpr uint32_t END_SKIP = 1u << 20, END_NOLIM = 1u << 21, END_LEV_I = 1u << 22, END_LEV_J = 1u << 23;

// fields of the two topology words of a local cell (local indices < 1024)
constexpr uint32_t TOPO_MOUTH = 0x7ff;         // word 0: downstream (11 bits), first upstream (10), flags (2)
constexpr int TOPO_UP0 = 11, TOPO_FLAGS = 21;
constexpr int TOPO_NUP = 10, TOPO_CODE = 18;   // word 1: second upstream (10 bits), upstream count (8), code (8)

// device copy of a plan
struct BlockTab {
    int T, kmax, nblk, closed;
    const int32_t* cell;
    const uint32_t* topo;
    const int32_t* upx_ptr;
    const uint16_t* upx;
    const int32_t* ndam;
    const int32_t* dom;
    int npth;                                  // > 0: blocks along paths with both ends in the network
    const int32_t* path;
    const uint32_t *pword, *pends, *pcell;
    const int32_t* ppx_ptr;
    const uint16_t* ppx;
    const double* pconst;                      // [5][nblk*T]: riverbeds of the ends, level elevation, width, distance
    int ndead;                                 // paths with an end outside the network, in dead
    const int32_t* dead;
};

// the arrays a launch hands to the next one: written by the owner of a cell while
// other blocks may still read the previous values
template <class R>
struct BlockState {
    double *rivsto, *fldsto, *levsto, *damsto;
    R *rivout, *fldout, *rivdph, *rivdph_pre, *fldsto_pre, *flddph, *fldfrc;
    R *pthflw, *levdph;                        // with paths
};

// Launches of an instance of nt substeps: one with a closed plan, else an even number
// of at most kmax substeps each, so that the state ends in the arrays it began in.
__host__ __device__ inline int block_launches(int nt, int kmax, int closed) {
    return closed ? 1 : 2 * ((nt + 2 * kmax - 1) / (2 * kmax));
}

// Launch j of an outer step: substeps nt*j/L .. nt*(j+1)/L of every instance with its
// own nt (S.inst) and L = block_launches(nt); instances with L <= j are done. S carries
// the values before it, O receives those after it (may alias S with a closed plan).
// I: the step of a single model. vel0: D2RIVOUT of the first substep where it differs
// from D2RIVOUT_PRE, or NULL. Budget sums of a single model go to
// S.partials[it][block][NPART].
template <class R>
hipError_t launch_block(const DevMap& M, const DevState<R>& S, const BlockState<R>& O, const BlockTab& P,
                        const StepArgs& A, const InstStep& I, int j, const R* vel0, hipStream_t st);

}  // namespace cmf
