// Device-side BSR pattern and element->BSR map (the TACS createSchurMat pattern the reference builds on the
// host, TestKernels.cpp:105, and generateElementBCSRMap, verification/TACSHelpers.h:138-182). Results are
// identical to the host builders in fem_host.cpp: block (i, j) exists iff nodes i and j share an element,
// columns sorted ascending, an isolated node keeps its diagonal block, map[e*N*N + i*N + j] = slot * bsize^2.
//
// Steps (all on one stream):
//   1. node -> element adjacency: per-node counts (atomics), exclusive scan, fill; each element's node ids
//      are also sorted once;
//   2. one thread per row merges the sorted lists of the row's (up to four) elements and counts the distinct
//      ids -> row lengths -> exclusive scan -> rowp. Rows of more elements go to a list that wavefronts work
//      through: they sort the row's node references in LDS (bitonic network);
//   3. the same again writes the distinct ids into cols;
//   4. the map: a workgroup copies the rows of a few elements to LDS and searches each (element, i, j) there
//      (elements of 4, 9, 16 or 25 nodes; else one thread per entry searches row i in global memory).
// Invalid node ids, rows with more candidates than a wavefront sorts, and map misses raise device flags
// that the host turns into status codes; no access depends on an unchecked id.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>
#include <vector>

#include "fem_amd.h"
#include "fem_internal.h"

namespace fem {
namespace {

#define FEM_HIP_CHECK(expr)                                                                               \
  do {                                                                                                    \
    hipError_t err_ = (expr);                                                                             \
    if (err_ != hipSuccess) {                                                                             \
      return set_error(FEM_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(err_), __FILE__,    \
                       __LINE__);                                                                         \
    }                                                                                                     \
  } while (0)

constexpr int kThreads = 256;
constexpr int kRowCap = 1024;  // candidates one wavefront sorts (node references of a row's elements)
constexpr int kScanItems = 4;  // items per thread in the block scan

constexpr int kMergeRows = 128;  // rows (threads) per workgroup of the merge
constexpr int kMergeLists = 4;   // elements of a row that the merge takes
constexpr int kMergeNodes = 32;  // nodes per element up to which the merge is used

// Device flags: [0] invalid node id, [1] row beyond kRowCap, [2] map miss, [3] pattern beyond 2^31 blocks; then
// [4] the pattern's blocks and [5] the rows left to the wavefront sort.
enum Flag { kBadNode = 0, kBigRow = 1, kMiss = 2, kOverflow = 3, kTotal = 4, kLongRows = 5, kFlags = 8 };

// Reference counts per node and (sorted != NULL) each element's node ids in ascending order, element-major.
__global__ __launch_bounds__(kThreads) void count_refs(int numNodes, int numElements, int npe, const int *connPtr,
                                                       const int *conn, int *cnt, int *sorted, int *flags) {
  const int64_t k = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (k >= int64_t(numElements) * npe) return;
  const int e = int(k / npe), a = int(k - int64_t(e) * npe);
  const int *en = conn + int64_t(connPtr[e]);
  const int n = en[a];
  if (sorted) {
    int rank = 0;
    for (int b = 0; b < npe; b++) rank += en[b] < n || (en[b] == n && b < a);
    sorted[int64_t(e) * npe + rank] = n;
  }
  if (n < 0 || n >= numNodes) {
    flags[kBadNode] = 1;
    return;
  }
  atomicAdd(&cnt[n], 1);
}

// Exclusive scan of `in` (n entries) into `out` (n + 1 entries, out[n] = total), in three passes: block sums,
// a one-block scan of the block sums, block-local scans plus offsets. Totals are int64.
__global__ __launch_bounds__(kThreads) void scan_block_sums(const int *in, int64_t n, int64_t *blockSums) {
  __shared__ int64_t part[kThreads];
  const int64_t base = int64_t(blockIdx.x) * kThreads * kScanItems;
  int64_t s = 0;
  for (int i = 0; i < kScanItems; i++) {
    const int64_t k = base + int64_t(threadIdx.x) * kScanItems + i;
    if (k < n) s += in[k];
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off /= 2) {
    if (int(threadIdx.x) < off) part[threadIdx.x] += part[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) blockSums[blockIdx.x] = part[0];
}

// One block: exclusive scan of the block sums in place (any count, in chunks of kThreads).
__global__ __launch_bounds__(kThreads) void scan_sums(int64_t *blockSums, int64_t numBlocks) {
  __shared__ int64_t buf[kThreads];
  int64_t carry = 0;
  for (int64_t c = 0; c < numBlocks; c += kThreads) {
    const int64_t k = c + threadIdx.x;
    const int64_t v = k < numBlocks ? blockSums[k] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kThreads; off *= 2) {  // inclusive Hillis-Steele scan
      const int64_t t = int(threadIdx.x) >= off ? buf[threadIdx.x - off] : 0;
      __syncthreads();
      buf[threadIdx.x] += t;
      __syncthreads();
    }
    if (k < numBlocks) blockSums[k] = carry + buf[threadIdx.x] - v;
    const int64_t total = buf[kThreads - 1];
    __syncthreads();
    carry += total;
  }
}

template <typename OutT>
__global__ __launch_bounds__(kThreads) void scan_apply(const int *in, int64_t n, const int64_t *blockOffsets, OutT *out,
                                                      int *flags, int *total) {
  __shared__ int64_t buf[kThreads];
  const int64_t base = int64_t(blockIdx.x) * kThreads * kScanItems;
  int64_t v[kScanItems];
  int64_t s = 0;
  for (int i = 0; i < kScanItems; i++) {
    const int64_t k = base + int64_t(threadIdx.x) * kScanItems + i;
    v[i] = k < n ? in[k] : 0;
    s += v[i];
  }
  buf[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < kThreads; off *= 2) {
    const int64_t t = int(threadIdx.x) >= off ? buf[threadIdx.x - off] : 0;
    __syncthreads();
    buf[threadIdx.x] += t;
    __syncthreads();
  }
  int64_t run = blockOffsets[blockIdx.x] + buf[threadIdx.x] - s;
  for (int i = 0; i < kScanItems; i++) {
    const int64_t k = base + int64_t(threadIdx.x) * kScanItems + i;
    if (k <= n) {
      if (run > INT32_MAX) flags[kOverflow] = 1;
      out[k] = OutT(run);  // k == n writes the total
      if (k == n && total) *total = int(run);
    }
    run += v[i];
  }
}

__global__ __launch_bounds__(kThreads) void fill_adjacency(int numNodes, int numElements, int npe, const int *connPtr,
                                                           const int *conn, int *cursor, int *adj) {
  const int64_t k = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (k >= int64_t(numElements) * npe) return;
  const int e = int(k / npe), a = int(k - int64_t(e) * npe);
  const int n = conn[int64_t(connPtr[e]) + a];
  if (n < 0 || n >= numNodes) return;  // flagged by count_refs
  adj[atomicAdd(&cursor[n], 1)] = e;
}

// One thread per row of up to kMergeLists elements: merges their sorted node ids. WRITE = false stores the
// number of distinct ids in len[row] and lists the other rows in longRows; WRITE = true stores the ids at
// cols[rowp[row]...], staged in LDS (`capacity` ints) so that a workgroup's rows are written as one run. Bound by
// the scattered loads of the list heads, which a workgroup's neighbouring rows share in the L1: 500 x 500 order 2
// (1.0M rows, 16M ids) 33 us to count and 41 us to write, against 350 us per pass for a wavefront per row and a
// bitonic sort of its references (kept for the other rows).
template <bool WRITE>
__global__ __launch_bounds__(kMergeRows) void merge_rows(int numNodes, int npe, const int *sorted, const int *nptr,
                                                         const int *adj, int *len, int *longRows, const int *rowp,
                                                         int *cols, int capacity, int *flags) {
  extern __shared__ int staged[];
  const int base = int(blockIdx.x) * kMergeRows, row = base + int(threadIdx.x);
  int first = 0, ids = 0;
  bool stage = false;
  if (WRITE) {
    first = rowp[base];
    ids = rowp[min(base + kMergeRows, numNodes)] - first;
    stage = ids <= capacity;  // no room when rows that the merge leaves out are long: written directly
  }
  if (row < numNodes) {
    const int e0 = nptr[row], ne = nptr[row + 1] - e0;
    int *out = nullptr;
    if (WRITE) out = stage ? staged + (rowp[row] - first) : cols + rowp[row];
    if (ne == 0) {  // a node of no element: diagonal block only
      if (WRITE) out[0] = row;
      else len[row] = 1;
    } else if (ne > kMergeLists) {
      if (!WRITE) longRows[atomicAdd(&flags[kLongRows], 1)] = row;
    } else {
      int head[kMergeLists], at[kMergeLists], end[kMergeLists];
#pragma unroll
      for (int i = 0; i < kMergeLists; i++) {
        at[i] = i < ne ? adj[e0 + i] * npe : 0;
        end[i] = i < ne ? at[i] + npe : 0;
        head[i] = i < ne ? sorted[at[i]] : INT32_MAX;
      }
      int count = 0, last = -1;
      for (;;) {
        int m = head[0];
#pragma unroll
        for (int i = 1; i < kMergeLists; i++) m = min(m, head[i]);
        if (m == INT32_MAX) break;
        if (m != last) {
          if (WRITE) out[count] = m;
          count++;
          last = m;
        }
#pragma unroll
        for (int i = 0; i < kMergeLists; i++) {
          if (head[i] == m) {
            at[i]++;
            head[i] = at[i] < end[i] ? sorted[at[i]] : INT32_MAX;
          }
        }
      }
      if (!WRITE) len[row] = count;
    }
  }
  if (WRITE && stage) {  // (rows left to the wavefront sort are overwritten by it)
    __syncthreads();
    for (int i = threadIdx.x; i < ids; i += kMergeRows) cols[first + i] = staged[i];
  }
}

// One wavefront per row: sorted distinct node ids of the row's elements, by a sort of their node references.
// WRITE = false stores the count in len[row]; WRITE = true stores the ids at cols[rowp[row]...]. Returns through
// flags when the row has more than kRowCap candidates. list == NULL: rows 0..numNodes-1, one per wavefront; else
// the flags[kLongRows] rows of the list, strided over the grid's wavefronts.
template <bool WRITE>
__device__ __forceinline__ void sort_row(int row, int *s, int lane, int npe, const int *connPtr, const int *conn,
                                         const int *nptr, const int *adj, int *len, const int *rowp, int *cols,
                                         int *flags) {
  const int e0 = nptr[row], ne = nptr[row + 1] - e0;
  const int k = ne * npe;
  if (k > kRowCap) {
    if (lane == 0) flags[kBigRow] = 1;
    return;
  }
  if (k == 0) {  // isolated node: diagonal block only
    if (lane == 0) {
      if (WRITE) cols[rowp[row]] = row;
      else len[row] = 1;
    }
    return;
  }
  int size = 64;
  while (size < k) size *= 2;
  for (int i = lane; i < size; i += 64) {
    int v = INT32_MAX;
    if (i < k) {
      const int e = adj[e0 + i / npe];
      v = conn[int64_t(connPtr[e]) + i % npe];
    }
    s[i] = v;
  }
  __syncwarp();
  // Bitonic sort of s[0, size) ascending; each lane handles pairs (i, i ^ j) with i < i ^ j.
  for (int w = 2; w <= size; w *= 2) {
    for (int j = w / 2; j > 0; j /= 2) {
      for (int i = lane; i < size; i += 64) {
        const int p = i ^ j;
        if (p > i) {
          const int x = s[i], y = s[p];
          const bool up = (i & w) == 0;
          if ((x > y) == up) {
            s[i] = y;
            s[p] = x;
          }
        }
      }
      __syncwarp();
    }
  }
  // Distinct ids in order: entry i is kept iff it differs from entry i - 1 (entries past k are INT32_MAX).
  int count = 0;
  for (int c = 0; c < k; c += 64) {
    const int i = c + lane;
    const bool keep = i < k && (i == 0 || s[i] != s[i - 1]);
    const unsigned long long m = __ballot(keep);
    if (WRITE && keep) cols[rowp[row] + count + __popcll(m & ((1ull << lane) - 1))] = s[i];
    count += __popcll(m);
  }
  if (!WRITE && lane == 0) len[row] = count;
}

template <bool WRITE>
__global__ __launch_bounds__(kThreads) void row_columns(int numNodes, int npe, const int *connPtr, const int *conn,
                                                        const int *nptr, const int *adj, int *len, const int *rowp,
                                                        int *cols, const int *list, int *flags) {
  constexpr int WAVES = kThreads / 64;
  __shared__ int keys[WAVES][kRowCap];
  const int wave = int(threadIdx.x / 64), lane = int(threadIdx.x % 64);
  const int n = list ? flags[kLongRows] : numNodes;
  for (int i = int(blockIdx.x) * WAVES + wave; i < n; i += int(gridDim.x) * WAVES) {  // i is wave-uniform
    sort_row<WRITE>(list ? list[i] : i, keys[wave], lane, npe, connPtr, conn, nptr, adj, len, rowp, cols, flags);
    __syncwarp();  // the row's reads are done before the next row overwrites its keys
  }
}

__device__ __forceinline__ int find_col(const int *cols, int b, int e, int col) {
  while (b < e) {
    const int m = (b + e) / 2;
    if (cols[m] < col) b = m + 1;
    else e = m;
  }
  return b;
}

// The map, one thread per entry (elements of another number of nodes than element_map_staged takes). maxBlocks: the
// blocks whose bs2 entries each 32-bit offsets reach (0 where one block is too many); a larger pattern gets no map.
__global__ __launch_bounds__(kThreads) void element_map(int numRows, int numElements, int npe, const int *connPtr,
                                                        const int *conn, const int *rowp, const int *cols, int bs2,
                                                        int maxBlocks, int *map, int *flags) {
  const int64_t k = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t nn = int64_t(npe) * npe;
  if (rowp[numRows] > maxBlocks) {
    flags[kOverflow] = 1;
    return;
  }
  if (k >= int64_t(numElements) * nn) return;
  const int e = int(k / nn), ij = int(k - int64_t(e) * nn), i = ij / npe, j = ij - i * npe;
  const int *en = conn + connPtr[e];
  const int r = en[i], c = en[j];
  if (r < 0 || r >= numRows || c < 0 || c >= numRows) {
    flags[kBadNode] = 1;
    return;
  }
  const int b = rowp[r], end = rowp[r + 1];
  const int pos = find_col(cols, b, end, c);
  if (pos >= end || cols[pos] != c) {
    flags[kMiss] = 1;
    return;
  }
  map[k] = pos * bs2;
}

// The map of PER elements of NPE nodes per workgroup: their rows' columns are copied to LDS (CAP ints per row, 13/4
// of an element's nodes at least; longer rows are searched in global memory), then every entry is a binary search
// there. 500 x 500 order 2 (20M entries): 118 us; 148 with 32 KB tiles, 152 us with every search in global memory.
template <int NPE>
struct MapTile {
  static constexpr int CAP = ((NPE * 13 + 3) / 4) | 1;
  static constexpr int PER = 2560 / (NPE * (CAP + 3));  // about 10 KB: eight workgroups per CU hide the chain of loads
  static constexpr int ROWS = PER * NPE;
};
template <int NPE>
__global__ __launch_bounds__(kThreads) void element_map_staged(int numRows, int numElements, const int *connPtr,
                                                               const int *conn, const int *rowp, const int *cols,
                                                               int bs2, int maxBlocks, int *map, int *flags) {
  constexpr int CAP = MapTile<NPE>::CAP, PER = MapTile<NPE>::PER, ROWS = MapTile<NPE>::ROWS;
  __shared__ int node[ROWS], begin[ROWS], count[ROWS], col[ROWS * CAP];
  if (rowp[numRows] > maxBlocks) {
    flags[kOverflow] = 1;
    return;
  }
  const int64_t e0 = int64_t(blockIdx.x) * PER;
  const int rows = int(min(int64_t(PER), numElements - e0)) * NPE;
  for (int k = threadIdx.x; k < ROWS; k += kThreads) {
    int n = -1;
    if (k < rows) {
      n = conn[int64_t(connPtr[e0 + k / NPE]) + k % NPE];
      if (n < 0 || n >= numRows) flags[kBadNode] = 1;
    }
    const bool ok = n >= 0 && n < numRows;
    node[k] = n;
    begin[k] = ok ? rowp[n] : 0;
    count[k] = ok ? rowp[n + 1] - rowp[n] : -1;  // no row: nothing is looked up in it
  }
  __syncthreads();
#pragma unroll 8
  for (int k = threadIdx.x; k < ROWS * CAP; k += kThreads) {
    const int r = k / CAP, i = k % CAP;
    if (i < count[r]) col[k] = cols[begin[r] + i];
  }
  __syncthreads();
#pragma unroll 2
  for (int k = threadIdx.x; k < rows * NPE; k += kThreads) {
    const int r = k / NPE, c = node[r / NPE * NPE + k % NPE];
    const int n = count[r], b = begin[r];
    if (n < 0 || c < 0 || c >= numRows) continue;
    int lo = 0;
    bool hit;
    if (n <= CAP) {
      lo = find_col(col + r * CAP, 0, n, c);
      hit = lo < n && col[r * CAP + lo] == c;
    } else {
      lo = find_col(cols, b, b + n, c) - b;
      hit = lo < n && cols[b + lo] == c;
    }
    if (hit) map[e0 * NPE * NPE + k] = (b + lo) * bs2;
    else flags[kMiss] = 1;
  }
}

__global__ __launch_bounds__(kThreads) void fill_zero(int *p, int64_t n) {
  const int64_t k = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (k < n) p[k] = 0;
}

// Device scratch of one call, from a block that is kept per device (at most kKeptBytes, one; calls that overlap on a
// device allocate their own). Calls synchronise their stream before they return, so a kept block is idle; after an
// error, when work may still be queued, the block is freed (which waits for the device).
constexpr size_t kKeptBytes = size_t(256) << 20;
struct KeptBlock {
  void *p = nullptr;
  size_t bytes = 0;
  int device = 0;
};
std::mutex keptMu;
std::vector<KeptBlock> kept;  // idle blocks, at most one per device

struct Scratch {
  KeptBlock b;
  bool done = false;  // the call's work has finished
  int alloc(size_t bytes) {
    FEM_HIP_CHECK(hipGetDevice(&b.device));
    {
      std::lock_guard<std::mutex> lk(keptMu);
      for (size_t i = 0; i < kept.size(); i++) {
        if (kept[i].device == b.device && kept[i].bytes >= bytes) {
          b = kept[i];
          kept.erase(kept.begin() + long(i));
          return FEM_OK;
        }
      }
    }
    const hipError_t e = hipError_t(device_alloc(&b.p, bytes));
    if (e != hipSuccess) {
      b.p = nullptr;
      return set_error(FEM_ERR_HIP, "hipMalloc of %zu bytes of pattern scratch failed: %s", bytes, hipGetErrorString(e));
    }
    b.bytes = bytes;
    return FEM_OK;
  }
  ~Scratch() {
    if (!b.p) return;
    KeptBlock drop = b;
    if (done && b.bytes <= kKeptBytes) {
      std::lock_guard<std::mutex> lk(keptMu);
      size_t i = 0;
      while (i < kept.size() && kept[i].device != b.device) i++;
      if (i == kept.size()) {
        kept.push_back(b);
        drop.p = nullptr;
      } else if (kept[i].bytes < b.bytes) {
        std::swap(drop, kept[i]);
      }
    }
    if (drop.p) (void)hipFree(drop.p);
  }
};

unsigned grid_for(int64_t n) { return unsigned((n + kThreads - 1) / kThreads); }

// Block sums an exclusive scan of n entries (n + 1 outputs) needs.
int64_t scan_blocks(int64_t n) {
  const int64_t perBlock = int64_t(kThreads) * kScanItems;
  return (n + 1 + perBlock - 1) / perBlock;
}

// Exclusive scan of in[0, n) into out[0, n] (see the scan kernels), with scan_blocks(n) block sums in `sums`.
template <typename OutT>
int exclusive_scan(const int *in, int64_t n, OutT *out, int *flags, int *total, int64_t *sums, hipStream_t stream) {
  const int64_t blocks = scan_blocks(n);
  scan_block_sums<<<unsigned(blocks), kThreads, 0, stream>>>(in, n, sums);
  scan_sums<<<1, kThreads, 0, stream>>>(sums, blocks);
  scan_apply<OutT><<<unsigned(blocks), kThreads, 0, stream>>>(in, n, sums, out, flags, total);
  FEM_HIP_CHECK(hipGetLastError());
  return FEM_OK;
}

int report_flags(const int (&h)[kFlags]) {
  if (h[kBadNode]) return set_error(FEM_ERR_INVALID_ARGUMENT, "a node id is outside [0, numNodes)");
  if (h[kBigRow]) {
    return set_error(FEM_ERR_UNSUPPORTED, "a node's elements hold more than %d node references (use the host "
                     "pattern builder)", kRowCap);
  }
  if (h[kMiss]) return set_error(FEM_ERR_MAP_MISS, "an element node pair has no block in the pattern");
  if (h[kOverflow]) return set_error(FEM_ERR_INVALID_ARGUMENT, "pattern exceeds 2^31 blocks");
  return FEM_OK;
}

int check_flags(const int *dflags, hipStream_t stream, int *total) {
  int h[kFlags] = {};
  FEM_HIP_CHECK(hipMemcpyAsync(h, dflags, sizeof(h), hipMemcpyDeviceToHost, stream));
  FEM_HIP_CHECK(hipStreamSynchronize(stream));
  *total = h[kTotal];
  return report_flags(h);
}

}  // namespace
}  // namespace fem

using namespace fem;

// Scratch of fem_bsr_pattern_device_noalloc: one array per GPU, held by the process (64 MiB). Host code never
// uses the array's name as an address: each device's copy is reached through the address
// hipGetSymbolAddress gives on that device, looked up once per device (device_scratch).
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace fem {
namespace {

// Scratch of one pattern build: error flags, per-node reference counts (then the fill cursor, then the list of rows
// the merge leaves out), node->element offsets, the adjacency list, row lengths, the scans' block sums and the
// elements' sorted node ids (NULL: every row is sorted by a wavefront).
struct PatternScratch {
  int *flags, *cnt, *nptr, *adj, *len;
  int64_t *sums;
  int *sorted;
};

constexpr size_t kScratchAlign = 256;
size_t align_bytes(size_t n) { return (n + kScratchAlign - 1) / kScratchAlign * kScratchAlign; }

// Bytes of each scratch array of a build over numNodes nodes and refs node references, in PatternScratch order.
void pattern_scratch_sizes(int numNodes, int64_t refs, size_t (&bytes)[6]) {
  const size_t nodes1 = (size_t(numNodes) + 1) * sizeof(int);
  bytes[0] = kFlags * sizeof(int);
  bytes[1] = bytes[2] = bytes[4] = nodes1;
  bytes[3] = size_t(std::max<int64_t>(refs, 1)) * sizeof(int);
  bytes[5] = size_t(scan_blocks(numNodes)) * sizeof(int64_t);
}

size_t pattern_scratch_total(const size_t (&bytes)[6]) {
  size_t need = 0;
  for (size_t b : bytes) need += align_bytes(b);
  return need;
}

// Bytes of the elements' sorted node ids; 0 where the merge does not take elements of that many nodes.
size_t sorted_bytes(int64_t refs, int nodesPerElement) {
  return nodesPerElement <= kMergeNodes ? size_t(refs) * sizeof(int) : 0;
}

// The scratch arrays laid out from `base`, the sorted ids (if wanted) last.
PatternScratch pattern_scratch(void *base, const size_t (&bytes)[6], bool sorted) {
  unsigned char *p = static_cast<unsigned char *>(base);
  void *arr[7];
  for (int i = 0; i < 6; i++) {
    arr[i] = p;
    p += align_bytes(bytes[i]);
  }
  arr[6] = sorted ? p : nullptr;
  return PatternScratch{static_cast<int *>(arr[0]), static_cast<int *>(arr[1]),     static_cast<int *>(arr[2]),
                        static_cast<int *>(arr[3]), static_cast<int *>(arr[4]), static_cast<int64_t *>(arr[5]),
                        static_cast<int *>(arr[6])};
}

int check_pattern_args(int numNodes, int numElements, int nodesPerElement, const int *connPtr, const int *conn,
                       const int *rowp, const int64_t *numBlocks) {
  if (numNodes < 0 || numElements < 0 || nodesPerElement <= 0) {
    return set_error(FEM_ERR_INVALID_ARGUMENT, "negative size (numNodes=%d numElements=%d nodesPerElement=%d)",
                     numNodes, numElements, nodesPerElement);
  }
  if (!rowp || !numBlocks) return set_error(FEM_ERR_NULL_POINTER, "rowp/numBlocks is NULL");
  if (numElements > 0 && (!connPtr || !conn)) return set_error(FEM_ERR_NULL_POINTER, "connPtr/conn is NULL");
  if (int64_t(numElements) * nodesPerElement > INT32_MAX) {
    return set_error(FEM_ERR_UNSUPPORTED, "more than 2^31 element node references");
  }
  return FEM_OK;
}

// The pattern build of fem_bsr_pattern_device on caller-provided scratch (arguments already checked).
int pattern_build(int numNodes, int numElements, int nodesPerElement, const int *connPtr, const int *conn, int *rowp,
                  int *cols, int64_t colsCapacity, int64_t *numBlocks, hipStream_t stream, const PatternScratch &sc) {
  const int64_t refs = int64_t(numElements) * nodesPerElement;
  int *flags = sc.flags, *cnt = sc.cnt, *nptr = sc.nptr, *adj = sc.adj, *len = sc.len;
  // cleared with a fill kernel (scratch may be reused across calls; no memset nodes)
  fill_zero<<<1, kThreads, 0, stream>>>(flags, kFlags);
  fill_zero<<<grid_for(int64_t(numNodes) + 1), kThreads, 0, stream>>>(cnt, int64_t(numNodes) + 1);
  if (refs > 0) {
    count_refs<<<grid_for(refs), kThreads, 0, stream>>>(numNodes, numElements, nodesPerElement, connPtr, conn, cnt,
                                                        sc.sorted, flags);
  }
  int rc = exclusive_scan<int>(cnt, numNodes, nptr, flags, nullptr, sc.sums, stream);
  if (rc) return rc;
  // cursor = nptr (cnt is reused as the fill cursor). Invalid ids are counted and filled nowhere; as columns they
  // are only values, and the flag that count_refs raised ends the call before any is written out.
  FEM_HIP_CHECK(hipMemcpyAsync(cnt, nptr, size_t(numNodes) * sizeof(int), hipMemcpyDeviceToDevice, stream));
  if (refs > 0) {
    fill_adjacency<<<grid_for(refs), kThreads, 0, stream>>>(numNodes, numElements, nodesPerElement, connPtr, conn, cnt,
                                                            adj);
  }
  // Rows: merged (the rest listed in cnt, whose cursors are no longer needed), or all sorted by wavefronts.
  const unsigned rowBlocks = unsigned((int64_t(numNodes) + kThreads / 64 - 1) / (kThreads / 64));
  const unsigned longBlocks = std::min(rowBlocks, 2048u);
  const unsigned mergeBlocks = unsigned((int64_t(numNodes) + kMergeRows - 1) / kMergeRows);
  if (numNodes > 0 && sc.sorted) {
    merge_rows<false><<<mergeBlocks, kMergeRows, 0, stream>>>(numNodes, nodesPerElement, sc.sorted, nptr, adj, len, cnt,
                                                             nullptr, nullptr, 0, flags);
    row_columns<false><<<longBlocks, kThreads, 0, stream>>>(numNodes, nodesPerElement, connPtr, conn, nptr, adj, len,
                                                           nullptr, nullptr, cnt, flags);
  } else if (numNodes > 0) {
    row_columns<false><<<rowBlocks, kThreads, 0, stream>>>(numNodes, nodesPerElement, connPtr, conn, nptr, adj, len,
                                                          nullptr, nullptr, nullptr, flags);
  }
  rc = exclusive_scan<int>(len, numNodes, rowp, flags, flags + kTotal, sc.sums, stream);
  if (rc) return rc;
  FEM_HIP_CHECK(hipGetLastError());
  int total = 0;
  rc = check_flags(flags, stream, &total);
  if (rc) return rc;
  *numBlocks = total;
  if (cols && total > colsCapacity) {
    return set_error(FEM_ERR_INVALID_ARGUMENT, "cols holds %lld entries, the pattern has %d blocks",
                     (long long)colsCapacity, total);
  }
  if (cols && numNodes > 0) {
    if (sc.sorted) {
      // LDS for rows of the usual length: (2p + 1)^2 ids where four elements meet, 13/4 of an element's nodes at most
      const int capacity = std::min(kMergeRows * nodesPerElement * 13 / 4, 16384);
      merge_rows<true><<<mergeBlocks, kMergeRows, size_t(capacity) * sizeof(int), stream>>>(
          numNodes, nodesPerElement, sc.sorted, nptr, adj, nullptr, cnt, rowp, cols, capacity, flags);
      row_columns<true><<<longBlocks, kThreads, 0, stream>>>(numNodes, nodesPerElement, connPtr, conn, nptr, adj,
                                                            nullptr, rowp, cols, cnt, flags);
    } else {
      row_columns<true><<<rowBlocks, kThreads, 0, stream>>>(numNodes, nodesPerElement, connPtr, conn, nptr, adj,
                                                           nullptr, rowp, cols, nullptr, flags);
    }
    FEM_HIP_CHECK(hipGetLastError());
    FEM_HIP_CHECK(hipStreamSynchronize(stream));
  }
  return FEM_OK;
}

std::mutex scratchMu;
std::vector<void *> scratchAddr;  // per device ordinal; NULL until looked up

int device_scratch(void **out) {
  int dev = 0;
  FEM_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(scratchMu);
  if (dev >= int(scratchAddr.size())) scratchAddr.resize(size_t(dev) + 1, nullptr);
  if (!scratchAddr[size_t(dev)]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      return set_error(FEM_ERR_HIP, "hipGetSymbolAddress of the pattern scratch failed on device %d: %s", dev,
                       hipGetErrorString(e));
    }
    scratchAddr[size_t(dev)] = p;
  }
  *out = scratchAddr[size_t(dev)];
  return FEM_OK;
}

}  // namespace
}  // namespace fem

extern "C" int fem_bsr_pattern_device(int numNodes, int numElements, int nodesPerElement, const int *connPtr,
                                      const int *conn, int *rowp, int *cols, int64_t colsCapacity, int64_t *numBlocks,
                                      void *streamPtr) {
  int rc = check_pattern_args(numNodes, numElements, nodesPerElement, connPtr, conn, rowp, numBlocks);
  if (rc) return rc;
  hipStream_t stream = static_cast<hipStream_t>(streamPtr);
  size_t bytes[6];
  const int64_t refs = int64_t(numElements) * nodesPerElement;
  pattern_scratch_sizes(numNodes, refs, bytes);
  Scratch sc;
  rc = sc.alloc(pattern_scratch_total(bytes) + sorted_bytes(refs, nodesPerElement));
  if (rc) return rc;
  rc = pattern_build(numNodes, numElements, nodesPerElement, connPtr, conn, rowp, cols, colsCapacity, numBlocks, stream,
                     pattern_scratch(sc.b.p, bytes, sorted_bytes(refs, nodesPerElement) > 0));
  sc.done = rc == FEM_OK;
  return rc;
}

extern "C" int fem_bsr_pattern_device_noalloc(int numNodes, int numElements, int nodesPerElement, const int *connPtr,
                                              const int *conn, int *rowp, int *cols, int64_t colsCapacity,
                                              int64_t *numBlocks, void *streamPtr) {
  int rc = check_pattern_args(numNodes, numElements, nodesPerElement, connPtr, conn, rowp, numBlocks);
  if (rc) return rc;
  size_t bytes[6];
  const int64_t refs = int64_t(numElements) * nodesPerElement;
  pattern_scratch_sizes(numNodes, refs, bytes);
  const size_t need = pattern_scratch_total(bytes), extra = sorted_bytes(refs, nodesPerElement);
  if (need > kNoAllocScratchBytes) {
    return set_error(FEM_ERR_INVALID_ARGUMENT, "the pattern of %d nodes and %lld node references needs %zu bytes of "
                     "scratch; fem_bsr_pattern_device_noalloc holds %zu (use fem_bsr_pattern_device)", numNodes,
                     (long long)refs, need, kNoAllocScratchBytes);
  }
  void *base = nullptr;
  rc = device_scratch(&base);
  if (rc) return rc;
  // the merge of sorted lists where they fit the array too, else the wavefront sort
  return pattern_build(numNodes, numElements, nodesPerElement, connPtr, conn, rowp, cols, colsCapacity, numBlocks,
                       static_cast<hipStream_t>(streamPtr),
                       pattern_scratch(base, bytes, extra > 0 && need + extra <= kNoAllocScratchBytes));
}

extern "C" int fem_element_bcsr_map_device(const int *connPtr, const int *conn, int numElements, int nodesPerElement,
                                           int numRows, const int *rowp, const int *cols, int bsize, int *map,
                                           void *streamPtr) {
  if (numRows < 0 || numElements < 0 || nodesPerElement <= 0) {
    return set_error(FEM_ERR_INVALID_ARGUMENT, "negative size (numRows=%d numElements=%d nodesPerElement=%d)",
                     numRows, numElements, nodesPerElement);
  }
  if (bsize < 1) return set_error(FEM_ERR_INVALID_ARGUMENT, "bsize %d < 1", bsize);
  if (numElements == 0) return FEM_OK;
  if (!connPtr || !conn || !rowp || !cols || !map) {
    return set_error(FEM_ERR_NULL_POINTER, "connPtr/conn/rowp/cols/map is NULL");
  }
  hipStream_t stream = static_cast<hipStream_t>(streamPtr);
  Scratch sc;
  int rc = sc.alloc(kFlags * sizeof(int));
  if (rc) return rc;
  int *flags = static_cast<int *>(sc.b.p);
  const int64_t entries = int64_t(bsize) * bsize;  // of a block: beyond 32 bits from bsize 46341 on
  const int maxBlocks = int(INT32_MAX / entries), bs2 = int(std::min<int64_t>(entries, INT32_MAX));
  fill_zero<<<1, kThreads, 0, stream>>>(flags, kFlags);
  auto staged = [&](auto npe) {
    constexpr int NPE = decltype(npe)::value, PER = MapTile<NPE>::PER;
    element_map_staged<NPE><<<unsigned((int64_t(numElements) + PER - 1) / PER), kThreads, 0, stream>>>(
        numRows, numElements, connPtr, conn, rowp, cols, bs2, maxBlocks, map, flags);
  };
  switch (nodesPerElement) {
    case 4: staged(std::integral_constant<int, 4>{}); break;
    case 9: staged(std::integral_constant<int, 9>{}); break;
    case 16: staged(std::integral_constant<int, 16>{}); break;
    case 25: staged(std::integral_constant<int, 25>{}); break;
    default: {
      const int64_t n = int64_t(numElements) * nodesPerElement * nodesPerElement;
      element_map<<<grid_for(n), kThreads, 0, stream>>>(numRows, numElements, nodesPerElement, connPtr, conn, rowp,
                                                        cols, bs2, maxBlocks, map, flags);
    }
  }
  FEM_HIP_CHECK(hipGetLastError());
  int h[kFlags] = {};
  FEM_HIP_CHECK(hipMemcpyAsync(h, flags, sizeof(h), hipMemcpyDeviceToHost, stream));
  FEM_HIP_CHECK(hipStreamSynchronize(stream));
  sc.done = true;
  if (h[kOverflow]) {  // nothing was written
    return set_error(FEM_ERR_UNSUPPORTED, "the pattern's blocks x %lld entries overflow the map's 32-bit offsets",
                     (long long)entries);
  }
  return report_flags(h);
}

int fem::pattern_scratch_clear() {
  std::lock_guard<std::mutex> lk(keptMu);
  const int n = int(kept.size());
  for (const KeptBlock &b : kept) (void)hipFree(b.p);
  kept.clear();
  return n;
}

int fem::device_alloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess && pattern_scratch_clear() > 0) {
    (void)hipGetLastError();
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) (void)hipGetLastError();
  return int(e);
}
