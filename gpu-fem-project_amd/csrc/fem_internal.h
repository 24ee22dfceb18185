// Internal declarations shared by the host code (fem_host.cpp) and the HIP code (fem_device.hip).
#pragma once

#include <cstdint>
#include <vector>

#include "fem_amd.h"

namespace fem {

// Records `code` and a printf-style message as the calling thread's last error; returns `code`.
int set_error(int code, const char *fmt, ...);
void clear_error();

constexpr int nodes_per_element(int order) { return (order + 1) * (order + 1); }
// Bytes of column rank stored per (element, column node): N rounded up to whole 32-bit words.
constexpr int rank_pad(int order) { return (nodes_per_element(order) + 3) / 4 * 4; }

// Launch geometry of the owner-computes kernel, shared by the host partitioner (which sizes parts
// to fit) and the kernel templates (which size their LDS from it).
//   waves     wavefronts per workgroup
//   maxBlocks BSR blocks a part may own (FP64 LDS accumulator, 32 B per block)
//   maxRows   block rows a part may own
//   maxVisits element visits per part (waves x elements per wavefront: one batch per wave)
struct OwnerConfig {
  int waves;
  int maxBlocks;
  int maxRows;
  int maxVisits;
};
// Orders 1-2: one workgroup of 8 waves per CU (two per SIMD) sharing an accumulator of 2720 FP64 blocks,
// so parts are twice as large as with two 4-wave workgroups and fewer elements are visited twice
// (1.45 visits per element at 1000x1000 order 2; along a Morton curve 1.53, against 1.83 for the smaller parts).
// Orders 3-4: two workgroups of 4 waves per CU, each with half the LDS.
constexpr OwnerConfig owner_config(int order) {
  return order == 1   ? OwnerConfig{8, 2720, 352, 128}
         : order == 2 ? OwnerConfig{8, 2720, 320, 56}
         : order == 3 ? OwnerConfig{4, 1312, 96, 16}
                      : OwnerConfig{4, 1312, 64, 8};
}
// Residual-only parts: only the per-row residual lives in LDS. Deterministic plans take up to kResidualOnlyMaxRows
// rows per part; the others (line kernel) residual_rows(order): larger parts visit fewer elements twice, smaller
// ones fill the chip better (701 x 699 elements, us at 1024 / 768 / 512 / 320 rows: order 1 23.2 / 24.0 / 22.3 /
// 21.7, order 2 56.8 / 54.6 / 53.8 / 58.7, order 3 150 / 130 / 143 / 166, order 4 335 / 376 / 472 / 482). Meshes
// too small for a part per CU take smaller parts, down to 128 rows (30 x 33, order 4: 17.0 us at 1024 rows, 10.8
// at 320).
constexpr int kResidualOnlyMaxRows = 1024;
constexpr int residual_rows(int order) { return order <= 2 ? 512 : order == 3 ? 768 : kResidualOnlyMaxRows; }
constexpr int kNoRow = 0xffff;  // PlanHost::visitRow of a node another part owns

// Host-side result of partitioning a mesh into owner parts.
struct PlanHost {
  int order = 0;
  int numNodes = 0;
  int numElements = 0;
  int numParts = 0;
  int numColours = 1;
  int maxRowLength = 0;
  int64_t numBlocks = 0;
  std::vector<int> visitConn;     // [visits*N] nodes of each element visit (parts' visits contiguous)
  std::vector<int> visitEid;      // [visits] element id of each visit
  std::vector<uint16_t> visitRow; // [visits*N] residual-only plans of the line kernel: the node's part row, or kNoRow
  std::vector<int> nodeLrow;      // [numNodes] index of the node within its part's row list
  std::vector<int> partRowPtr;    // [P+1]
  std::vector<int> rows;          // global row (node) ids, ascending within a part
  std::vector<int> rowLbase;      // LDS block offset of each owned row within its part
  std::vector<int> partBlocks;    // [P] blocks owned by the part
  std::vector<int> partRunPtr;    // [P+1]
  std::vector<int> runs;          // [R*4] (lds block start, global block start, blocks, 0)
  std::vector<int> partElemPtr;   // [P+1] visit range of each part; visits grouped by colour
  std::vector<int> colourOff;     // [P*(C+1)] offsets of each colour within a part's visit list
  std::vector<uint8_t> rank;      // [E][N][rank_pad] rank[e][j][i]: slot of column conn[e,j] in row conn[e,i]
  std::vector<int> partDesc;      // [P*8] (first row, rows, blocks, first run, runs, first visit, visits, 0)
  int maxPartVisits = 0, maxPartRows = 0;
};

// Element-once tables (orders 3-4). Every output (a BSR block, or a node's residual pair) is either
// exclusive, formed by exactly one (element, node[, node]) contribution, or not. The contributions to any other
// output have slots, grouped by output, and the output is the sum of its slots in slot order (zero when no element
// touches it), so the result is bitwise reproducible. Plans keep these tables in the form of GatherList.
struct SplitHost {
  std::vector<int> code;   // [E][N][N], row-major (a, b): block of rows conn[e,a] x column conn[e,b]; below
                           // numBlocks the block's BSR index (exclusive), else numBlocks + staging slot
  std::vector<int> rcode;  // [E][N]: conn[e,a] if the node's residual is exclusive, else numNodes + slot
  std::vector<int> dst;    // BSR indices of the non-exclusive blocks, ascending
  std::vector<int> ptr;    // [dst.size() + 1] slot range of each
  std::vector<int> rdst;   // non-exclusive residual nodes, ascending
  std::vector<int> rptr;   // [rdst.size() + 1]
  int64_t slots = 0, rslots = 0;
};

// Builds the element-once tables from the connectivity ([E][N], element-major), the BSR row starts and a
// plan's column ranks. Returns FEM_ERR_UNSUPPORTED if the codes would not fit in an int.
int build_split_host(int order, int numNodes, int numElements, const int *conn, const int *rowp,
                     const std::vector<uint8_t> &rank, int64_t numBlocks, SplitHost &out);

// What a plan's element-once assembly does with those tables. An output's first contribution is stored in place,
// like an exclusive one; the others go to staging slots, numbered in contribution order (so an element's are
// contiguous), and the gather adds them. It works on lines of 64 bytes of the output array (unitsPerLine
// outputs each) that hold at least one output to add to: line l's unit u is output unitsPerLine * line[l] + u and
// gets the slots src[ptr[unitsPerLine * l + u]] .. src[ptr[unitsPerLine * l + u + 1] - 1] added in that
// order; a slot of -1 stands for an output without contributions, which is stored as zero.
struct GatherList {
  std::vector<int> line, ptr, src;
  int64_t slots = 0;
};
// Rewrites code (destinations below `outputs`, else outputs + slot; dst / ptr as in SplitHost) accordingly.
void plan_gather(int64_t outputs, int unitsPerLine, std::vector<int> &code, const std::vector<int> &dst,
                 const std::vector<int> &ptr, GatherList &out);

// partScale (0, 1] scales the part budgets (blocks, rows, visits) below the kernel's maxima: smaller
// parts give small meshes more workgroups at the price of more elements recomputed on part boundaries.
int build_plan_host(int order, int numNodes, int numElements, const int *connPtr, const int *conn,
                    const int *rowp, const int *cols, const double *nodeCoords, int flags, PlanHost &out,
                    double partScale = 1.0);

// Frees the idle scratch that the device pattern and map builders keep (fem_pattern.hip); returns the blocks freed.
int pattern_scratch_clear();
// hipMalloc for all of the library's device memory: where there is no room it first frees that scratch. Returns the
// hipError_t and leaves no error pending.
int device_alloc(void **p, size_t bytes);

// Batches (fem_device.hip). Doubles of element-once staging a Jacobian job of `plan` takes (0: the plan has no
// element-once tables); fem_batch_add with that staging owned by the caller (`stage`, NULL: the batch's own
// arena, grown at assembly); whether a plan's parts fit the streaming kernel (graph batches need it).
int64_t batch_stage_doubles(const fem_plan *plan, bool withResidual);
int batch_add_staged(fem_batch *batch, fem_plan *plan, const double *states, const double *nodeCoords, double E,
                     double nu, double t, double *residual, double *matEntries, double *stage);
bool plan_streams_public(const fem_plan *plan);
// For a FEM_BATCH_GRAPH batch that was never assembled, the server's: launches every group's kernels once with no work,
// records graphs of the server's full composition (residual-only and residual + Jacobian jobs of all orders; other
// compositions are launched directly) and replays them with no work. The runtime's first-launch allocations (code,
// scratch of kernels that spill, graph arguments) happen now, and none while serving. No-op without FEM_BATCH_GRAPH.
int batch_prepare(fem_batch *batch, int precision);
// fem_plan_assemble (accumulate false) and fem_plan_assemble_accumulate (true).
int plan_assemble(fem_plan *plan, const double *states, const double *nodeCoords, double E, double nu, double t,
                  double *residual, double *matEntries, int precision, void *stream, double *elapsedSeconds,
                  bool accumulate);

}  // namespace fem

// Opaque plan handle (device-resident arrays built from a PlanHost).
struct fem_plan {
  int order = 0;
  int numNodes = 0;
  int numElements = 0;
  int numParts = 0;
  int numColours = 1;
  int flags = 0;
  int device = 0;
  int64_t numBlocks = 0;
  int64_t elementVisits = 0;
  int64_t deviceBytes = 0;
  int *dVisitConn = nullptr;
  int *dVisitEid = nullptr;
  uint16_t *dVisitRow = nullptr;
  int *dNodeLrow = nullptr;
  int *dRows = nullptr;
  int *dRowLbase = nullptr;
  int *dRuns = nullptr;
  int *dColourOff = nullptr;
  int *dPartDesc = nullptr;
  uint8_t *dRank = nullptr;
  // Element-once assembly of Jacobian plans of orders 3-4 (SplitHost): connectivity, codes, gather lists and
  // staging arrays. dConn is NULL when the plan has none.
  int *dConn = nullptr;      // [E][N]
  int *dCode = nullptr;      // [E][N][N]
  int *dRcode = nullptr;     // [E][N]
  int *dGline = nullptr, *dGptr = nullptr, *dGsrc = nullptr;  // GatherList of the blocks (2 per line)
  int *dRline = nullptr, *dRptr = nullptr, *dRsrc = nullptr;  // and of the residual entries (4 per line)
  double *dStage = nullptr;  // [4 * slots]
  double *dRstage = nullptr; // [2 * rslots]
  int numGather = 0, numRgather = 0;    // gathered lines
  int64_t numSlots = 0, numRslots = 0;  // staged contributions: blocks, residual entries
  double partScale = 1.0;    // part budgets relative to the kernel's (FEM_PLAN_AUTOTUNE picks it)
  double tunedSeconds = 0;   // measured assembly time of the chosen build (autotuned plans)
  int tiledWaves = 4;        // orders 3-4: wavefronts per workgroup of the element-once kernel (autotuned)
  int maxPartVisits = 0, maxPartRows = 0;
  int numCUs = 0;
};
