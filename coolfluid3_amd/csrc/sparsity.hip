// Device construction of the LSS sparsity and of the element scatter structures.
//
// Node graph: plugins/UFEM/src/UFEM/SparsityBuilder.cpp:157-189 (per node the sorted set of all nodes
// sharing an element with it, self included).  Here: all element node pairs are encoded as
// row*N + col, radix-sorted and de-duplicated; row starts come from binary searches, so the result
// is independent of thread scheduling (bit-exact with the set-based construction).
//
// Element-to-slot map: block slot of (e, a, b) = position of conn[e][b] in row conn[e][a]
// (what TrilinosFEVbrMatrix::add_values finds by linear search, TrilinosFEVbrMatrix.cpp:330-352).
//
// Row-owner scatter structures used by the assembly kernel:
//   inc_ptr/inc     node -> incident (element, local node) pairs, sorted by element
//   wg_rows         node-row ranges handled by one assembly workgroup
//   inc_pos/blk_beg staging maps.  Within a workgroup, the element blocks of one staging pass are
//                   written to LDS rows sorted by (CSR block slot, incidence): the block of incidence
//                   q and column local node b goes to row inc_pos[q][b]; the rows of block s in pass
//                   p are [blk_beg[s][p], blk_beg[s+1][p]).  Simplices stage one pass per column
//                   local node b (p = b); Q1 cells (hexahedra, quadrilaterals) stage all (q, b) at once.
//   blk_acc         accumulator threads of each block (first index within the workgroup, count):
//                   c threads share the rows of a block (thread h takes rows h, h+c, ...) so that no
//                   thread sums more than kAccRows rows per pass; their partial sums are added in
//                   thread order when the block is written.
//   The maps come from the per-slot contribution lists sorted by (slot, b, q): the summation order is
//   fixed, so results are deterministic and no floating-point atomics are used.
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "internal.hpp"

namespace cf3hip {

namespace {

constexpr uint32_t kAccRows = 2;   // staged rows one accumulator thread sums per pass (at most)

int bits_for(uint64_t v)
{
  int b = 0;
  while(b < 64 && (v >> b) != 0) ++b;
  return std::max(b, 1);
}

__global__ void k_pair_keys(const uint32_t* __restrict__ conn, uint32_t n_elems, int k, uint64_t N,
                            uint64_t* __restrict__ keys)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t total = (uint64_t)n_elems * k * k;
  if(t >= total) return;
  const uint64_t e = t / (k * k);
  const int ab = (int)(t % (k * k));
  const uint32_t ra = conn[e * k + ab / k];
  const uint32_t cb = conn[e * k + ab % k];
  keys[t] = (uint64_t)ra * N + cb;
}

__device__ inline uint64_t lower_bound64(const uint64_t* a, uint64_t n, uint64_t v)
{
  uint64_t lo = 0, hi = n;
  while(lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if(a[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__device__ inline uint32_t lower_bound32(const uint32_t* a, uint32_t lo, uint32_t hi, uint32_t v)
{
  while(lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if(a[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__global__ void k_row_ptr_from_keys(const uint64_t* __restrict__ keys, uint64_t n, uint64_t N, uint64_t stride,
                                    uint32_t* __restrict__ row_ptr)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(i > N) return;
  row_ptr[i] = (uint32_t)lower_bound64(keys, n, i * stride);
}

__global__ void k_cols_from_keys(const uint64_t* __restrict__ keys, uint64_t n, uint64_t N, uint32_t* __restrict__ cols)
{
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(j >= n) return;
  cols[j] = (uint32_t)(keys[j] % N);
}

__global__ void k_slots(const uint32_t* __restrict__ conn, uint32_t n_elems, int k, const uint32_t* __restrict__ row_ptr,
                        const uint32_t* __restrict__ cols, uint32_t* __restrict__ slots)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t total = (uint64_t)n_elems * k * k;
  if(t >= total) return;
  const uint64_t e = t / (k * k);
  const int ab = (int)(t % (k * k));
  const uint32_t ra = conn[e * k + ab / k];
  const uint32_t cb = conn[e * k + ab % k];
  slots[t] = lower_bound32(cols, row_ptr[ra], row_ptr[ra + 1], cb);
}

__global__ void k_diag_blocks(uint32_t N, const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ cols,
                              uint32_t* __restrict__ diag)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= N) return;
  const uint32_t q = lower_bound32(cols, row_ptr[i], row_ptr[i + 1], i);
  diag[i] = (q < row_ptr[i + 1] && cols[q] == i) ? q : 0xffffffffu;
}

__global__ void k_inc_keys(const uint32_t* __restrict__ conn, uint64_t nek, uint64_t* __restrict__ keys)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(t >= nek) return;
  keys[t] = (uint64_t)conn[t] * nek + t;
}

__global__ void k_inc_from_keys(const uint64_t* __restrict__ keys, uint64_t nek, uint32_t* __restrict__ inc)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(t >= nek) return;
  inc[t] = (uint32_t)(keys[t] % nek);
}

// contribution key: slot * 2^16 + b * 2^12 + q (a row with more incidences than q has bits is refused below)
__global__ void k_contrib_keys(const uint32_t* __restrict__ conn, const uint32_t* __restrict__ inc,
                               const uint32_t* __restrict__ inc_ptr, const uint32_t* __restrict__ slots,
                               uint64_t nek, int k, uint64_t* __restrict__ keys)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(t >= nek) return;
  const uint32_t ea = inc[t];
  const uint32_t row = conn[ea];
  const uint32_t q = min((uint32_t)(t - inc_ptr[row]), 4095u);
  for(int b = 0; b < k; ++b) {
    const uint64_t s = slots[(uint64_t)ea * k + b];
    keys[t * k + b] = (s << 16) | ((uint64_t)b << 12) | q;
  }
}

__global__ void k_contrib_from_keys(const uint64_t* __restrict__ keys, uint64_t n, uint16_t* __restrict__ contrib)
{
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(j >= n) return;
  const uint64_t key = keys[j];
  const uint32_t b = (uint32_t)((key >> 12) & 15);
  const uint32_t q = (uint32_t)(key & 4095);
  contrib[j] = (uint16_t)((q << 4) | b);
}

// The block lists of one block, in order: groups of contributions with the same column mesh node (one group
// unless the system is periodic), each split evenly over ceil(n / len) lists.  contrib: (q << 4 | b) in
// (b, q) order, q relative to the block's row, whose incidences start at inc_row.  emit(at, count) is called
// per list; at(m) is the position of its contribution m.
template<class F>
__device__ inline void for_block_lists(const uint16_t* contrib, uint32_t n, bool periodic, int k, uint32_t len,
                                       const uint32_t* inc_row, const uint32_t* conn, F emit)
{
  if(!periodic) {
    const uint32_t nl = (n + len - 1) / len;
    for(uint32_t l = 0; l < nl; ++l) {
      const uint32_t i0 = (n * l) / nl, i1 = (n * (l + 1)) / nl;   // at most len
      emit([&](uint32_t m) { return i0 + m; }, i1 - i0);
    }
    return;
  }
  auto node = [&](uint32_t j) {
    const uint32_t ea = inc_row[contrib[j] >> 4];
    return conn[ea - ea % (uint32_t)k + (contrib[j] & 15u)];
  };
  uint32_t idx[8];
  for(uint32_t j = 0; j < n; ++j) {
    const uint32_t nd = node(j);
    bool seen = false;
    for(uint32_t i = 0; i < j && !seen; ++i) seen = node(i) == nd;
    if(seen) continue;
    uint32_t size = 0;
    for(uint32_t i = j; i < n; ++i) size += node(i) == nd ? 1u : 0u;
    const uint32_t nl = (size + len - 1) / len;
    uint32_t i = j;
    for(uint32_t l = 0; l < nl; ++l) {
      const uint32_t take = (size * (l + 1)) / nl - (size * l) / nl;
      for(uint32_t m = 0; m < take; ++i)
        if(node(i) == nd) idx[m++] = i;
      emit([&](uint32_t m) { return idx[m]; }, take);
    }
  }
}

// Accumulator threads of a block: enough that none sums more than kAccRows staged rows per pass.
__global__ void k_block_acc(uint64_t n_blocks, int passes, const uint32_t* __restrict__ contrib_ptr,
                            const uint16_t* __restrict__ contrib, uint8_t* __restrict__ acc_cnt)
{
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(s >= n_blocks) return;
  uint32_t cnt[4] = {0, 0, 0, 0};
  for(uint32_t j = contrib_ptr[s]; j < contrib_ptr[s + 1]; ++j) ++cnt[passes == 1 ? 0 : (contrib[j] & 15u)];
  const uint32_t mx = max(max(cnt[0], cnt[1]), max(cnt[2], cnt[3]));
  acc_cnt[s] = (uint8_t)max(1u, (mx + kAccRows - 1) / kAccRows);
}

// Per row: accumulator threads of the staged reduction (low half) and block lists (high half; simplices,
// len > 0), each saturated at 0xffff (above any workgroup's limit).  A row of more incidences than a workgroup
// holds is refused by the caller: its lists are not counted.
__global__ void k_row_acc(uint32_t n, const uint32_t* __restrict__ row_ptr, const uint8_t* __restrict__ acc_cnt,
                          uint32_t len, bool periodic, int k, const uint32_t* __restrict__ contrib_ptr,
                          const uint16_t* __restrict__ contrib, const uint32_t* __restrict__ inc_ptr,
                          const uint32_t* __restrict__ inc, const uint32_t* __restrict__ conn,
                          uint32_t* __restrict__ row_acc)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  uint32_t a = 0, l = 0;
  const bool count = len > 0 && inc_ptr[i + 1] - inc_ptr[i] <= (uint32_t)kAsmThreads;
  for(uint32_t s = row_ptr[i]; s < row_ptr[i + 1]; ++s) {
    a += acc_cnt[s];
    if(!count) continue;
    const uint32_t c0 = contrib_ptr[s], nc = contrib_ptr[s + 1] - c0;
    if(!periodic) l += (nc + len - 1) / len;
    else for_block_lists(contrib + c0, nc, true, k, len, inc + inc_ptr[i], conn, [&](auto, uint32_t) { ++l; });
  }
  row_acc[i] = min(a, 0xffffu) | (min(l, 0xffffu) << 16);
}

// One workgroup per assembly workgroup: derive the staging maps from the contribution lists of its
// blocks (contrib_ptr/contrib, sorted by (slot, b, q)) and number its accumulator threads.
__global__ __launch_bounds__(kAsmThreads) void k_stage_maps(int passes, int pos_stride,
                                                            const uint32_t* __restrict__ wg_rows,
                                                            const uint32_t* __restrict__ row_ptr,
                                                            const uint32_t* __restrict__ inc_ptr,
                                                            const uint32_t* __restrict__ contrib_ptr,
                                                            const uint16_t* __restrict__ contrib,
                                                            const uint8_t* __restrict__ acc_cnt,
                                                            uint8_t* __restrict__ inc_pos, uint8_t* __restrict__ blk_beg,
                                                            uint16_t* __restrict__ blk_acc)
{
  __shared__ uint32_t s_cnt[5][kAsmThreads];
  const uint32_t r0 = wg_rows[blockIdx.x], r1 = wg_rows[blockIdx.x + 1];
  const uint32_t blk0 = row_ptr[r0], nblk = row_ptr[r1] - blk0;
  const uint32_t t = threadIdx.x;
  uint32_t cnt[4] = {0, 0, 0, 0};
  if(t < nblk)
    for(uint32_t j = contrib_ptr[blk0 + t]; j < contrib_ptr[blk0 + t + 1]; ++j)
      ++cnt[passes == 1 ? 0 : (contrib[j] & 15u)];
  for(int p = 0; p < 4; ++p) s_cnt[p][t] = cnt[p];
  s_cnt[4][t] = t < nblk ? acc_cnt[blk0 + t] : 0;
  __syncthreads();
  if(t < 5) {   // exclusive scans over the blocks: one per pass, and the accumulator numbering
    uint32_t run = 0;
    for(uint32_t j = 0; j < nblk; ++j) {
      const uint32_t c = s_cnt[t][j];
      s_cnt[t][j] = run;
      run += c;
    }
  }
  __syncthreads();
  if(t < nblk) {
    // row of block t: row_ptr[row] <= blk0 + t < row_ptr[row + 1]; q counts the incidences of that row
    uint32_t lo = r0, hi = r1;
    while(hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if(row_ptr[mid] <= blk0 + t) lo = mid; else hi = mid;
    }
    const uint32_t ib = inc_ptr[lo];
    uint32_t beg[4];
    for(int p = 0; p < 4; ++p) {
      beg[p] = s_cnt[p][t];
      blk_beg[(uint64_t)(blk0 + t) * 4 + p] = (uint8_t)beg[p];
    }
    blk_acc[blk0 + t] = (uint16_t)(s_cnt[4][t] | ((uint32_t)acc_cnt[blk0 + t] << 8));
    for(uint32_t j = contrib_ptr[blk0 + t]; j < contrib_ptr[blk0 + t + 1]; ++j) {
      const uint32_t c = contrib[j], b = c & 15u, q = c >> 4;
      const uint32_t p = passes == 1 ? 0 : b;
      inc_pos[(uint64_t)(ib + q) * pos_stride + b] = (uint8_t)(beg[p]++);
    }
  }
}

// ---- assembly plans of the specialised simplex kernels ----
// A plan is what one workgroup of assemble_lists_wg reads, at a fixed stride, so that all its loads but
// those of the node records start at once:
//   head   r0, rows, elements, nodes, blk0, blocks, block lists, 0
//   nodes  uint32[ns]: the distinct mesh nodes of its elements, ascending, the last one repeated
//   loc    uint32[128]: per element the local indices of its nodes, byte m = node m
//   lo     uint64[128], hi uint16[128]: the block lists, in block order.  Entry i (11 bits) = element << 4 |
//          a << 2 | b, the row and column local nodes; entries 0-4 at bits 11 i of lo, entry 5 in hi;
//          unused entries name element `elements`.  lo bits 55-62: local index of the column node, bit 63:
//          first list of a block; hi bit 15: first list of a row.
// All contributions of a list have the same column mesh node (under periodic links a block may have several).
// A workgroup takes consecutive rows while its distinct elements, lists and rows fit; element sharing between
// neighbouring rows is what makes a workgroup of elements cheaper than one of (element, row) incidences.

// Rows one wave partitions in order; a workgroup never spans two segments.  Long segments leave few short
// workgroups at their ends, short ones keep the partition of a small mesh from being one long chain.
inline uint32_t plan_segment(uint64_t rows) { return rows < 65536 ? 63 : 252; }

// Distance in rows from each incidence's row back to the nearest earlier row of its element (255: none
// within 254): the element is new to a workgroup that starts at r0 exactly when that row is before r0.
// Clears info[5], which the following kernels fill.
__global__ void k_inc_back(uint64_t nek, int k, const uint32_t* __restrict__ inc, const uint32_t* __restrict__ rconn,
                           uint8_t* __restrict__ back, uint32_t* __restrict__ info)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(t < 5) info[t] = 0;
  if(t >= nek) return;
  const uint32_t ea = inc[t], a = ea % (uint32_t)k;
  const uint32_t* en = rconn + (ea - a);
  const uint32_t row = en[a];
  uint32_t d = 255;
  for(uint32_t m = 0; m < (uint32_t)k; ++m) {
    // a periodic element may hold a row twice: its second node there is never new
    if(en[m] < row) d = min(d, row - en[m]);
    else if(en[m] == row && m < a) d = 0;
  }
  back[t] = (uint8_t)d;
}

// One wave per segment of rows: start[r] = 1 where a workgroup starts.  misfit becomes 1 when a row alone
// exceeds a limit.
__global__ __launch_bounds__(64) void k_plan_partition(uint32_t N, uint32_t segment, const uint32_t* __restrict__ inc_ptr,
                                                       const uint8_t* __restrict__ back,
                                                       const uint32_t* __restrict__ row_lists,
                                                       uint8_t* __restrict__ start, int* __restrict__ misfit)
{
  const uint32_t b = blockIdx.x * segment, e = min(N, b + segment);
  const uint32_t lane = threadIdx.x;
  uint32_t r0 = b, ne = 0, nl = 0;
  for(uint32_t r = b; r < e; ++r) {
    const uint32_t i0 = inc_ptr[r], i1 = inc_ptr[r + 1], lists = row_lists[r] >> 16;
    uint32_t fresh = 0, own = 0;   // elements new to the open workgroup, and to one that starts here
    for(uint32_t i = i0 + lane; i - lane < i1; i += 64) {
      const uint32_t d = i < i1 ? back[i] : 0;
      fresh += (uint32_t)__popcll(__ballot(i < i1 && d > r - r0));
      own += (uint32_t)__popcll(__ballot(i < i1 && d > 0));
    }
    if(own > kPlanElems || lists > (uint32_t)kAsmThreads) {
      if(lane == 0) misfit[0] = 1;
      return;
    }
    const bool open = r == b || ne + fresh > kPlanElems || nl + lists > (uint32_t)kAsmThreads ||
                      r - r0 >= (uint32_t)kAsmThreads;
    if(open) { r0 = r; ne = own; nl = lists; }
    else { ne += fresh; nl += lists; }
    if(lane == 0) start[r] = open ? 1 : 0;
  }
}

// ascending bitonic sort of S (a power of two) LDS values
template<uint32_t S>
__device__ inline void lds_sort(uint32_t* s, uint32_t t)
{
  for(uint32_t size = 2; size <= S; size <<= 1)
    for(uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for(uint32_t p = t; p < S / 2; p += kAsmThreads) {
        const uint32_t i = 2 * p - (p & (stride - 1)), j = i + stride;   // i has the stride bit clear
        const uint32_t a = s[i], b = s[j];
        if((a > b) == ((i & size) == 0)) { s[i] = b; s[j] = a; }
      }
      __syncthreads();
    }
}

// position of v in the ascending s[0, n), which holds it
__device__ inline uint32_t lds_find(const uint32_t* s, uint32_t n, uint32_t v)
{
  uint32_t lo = 0, hi = n;
  while(hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if(s[mid] <= v) lo = mid; else hi = mid;
  }
  return lo;
}

// exclusive scan of one value per thread; total in every thread
__device__ inline uint32_t wg_scan(uint32_t v, uint32_t* s_wave, uint32_t t, uint32_t& total)
{
  constexpr uint32_t W = kAsmThreads / 64;
  uint32_t x = v;
#pragma unroll
  for(uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if((t & 63u) >= off) x += y;
  }
  if((t & 63u) == 63u) s_wave[t >> 6] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for(uint32_t w = 0; w < W; ++w) {
    if(w < (t >> 6)) before += s_wave[w];
    total += s_wave[w];
  }
  __syncthreads();
  return before + x - v;
}

// slot of key in an open-addressing table of T (a power of two) LDS words, 0xffffffff = free; fresh is set
// for the one thread that put it there
template<uint32_t T>
__device__ inline uint32_t lds_insert(uint32_t* table, uint32_t key, bool& fresh)
{
  uint32_t h = (key * 2654435761u) >> 16;
  for(;; ++h) {
    h &= T - 1;
    const uint32_t old = atomicCAS(&table[h], 0xffffffffu, key);
    if(old == 0xffffffffu || old == key) { fresh = old != key; return h; }
  }
}

// The plan of one workgroup.  most[0..2]: largest node, element and list count seen; a plan with more than
// ns nodes is left unfinished (the caller runs again with more slots).
__global__ __launch_bounds__(kAsmThreads) void k_plan_fill(uint32_t N, uint32_t n_plan, int k, uint32_t len, bool periodic,
                                                           uint32_t ns, const uint32_t* __restrict__ wg_start,
                                                           const uint32_t* __restrict__ row_ptr,
                                                           const uint32_t* __restrict__ inc_ptr,
                                                           const uint32_t* __restrict__ inc,
                                                           const uint8_t* __restrict__ back,
                                                           const uint32_t* __restrict__ rconn,
                                                           const uint32_t* __restrict__ conn,
                                                           const uint32_t* __restrict__ contrib_ptr,
                                                           const uint16_t* __restrict__ contrib,
                                                           unsigned char* __restrict__ plans, uint32_t* __restrict__ most)
{
  constexpr uint32_t S = kAsmThreads * 4;   // at least the incidences of kPlanElems elements
  __shared__ uint32_t s_etab[2 * kAsmThreads], s_ntab[2 * kPlanNodes], s_uniq[kPlanNodes], s_wave[kAsmThreads / 64];
  __shared__ uint32_t s_elem[kAsmThreads], s_loc[kAsmThreads];
  __shared__ uint8_t s_eidx[2 * kAsmThreads];
  __shared__ uint16_t s_inc[S];             // per incidence: element << 2 | a
  __shared__ uint16_t s_contrib[4 * S];     // the contributions of the workgroup's blocks
  const uint32_t wg = blockIdx.x, t = threadIdx.x;
  const uint32_t r0 = wg_start[wg], r1 = wg + 1 < n_plan ? wg_start[wg + 1] : N;
  const uint32_t i0 = inc_ptr[r0], ninc = inc_ptr[r1] - i0;
  const uint32_t blk0 = row_ptr[r0], nblk = row_ptr[r1] - blk0;
  for(uint32_t j = t; j < 2 * kAsmThreads; j += kAsmThreads) s_etab[j] = 0xffffffffu;
  for(uint32_t j = t; j < 2 * kPlanNodes; j += kAsmThreads) s_ntab[j] = 0xffffffffu;
  __syncthreads();
  // distinct elements, in the order of their first incidence
  uint32_t ne = 0;
  for(uint32_t base = 0; base < ninc; base += kAsmThreads) {
    const uint32_t i = i0 + base + t;
    bool fresh = false, put;
    uint32_t ea = 0;
    if(base + t < ninc) {
      ea = inc[i];
      fresh = back[i] > rconn[ea] - r0;
    }
    uint32_t total;
    const uint32_t at = ne + wg_scan(fresh ? 1u : 0u, s_wave, t, total);
    if(fresh) {
      s_elem[at] = ea / (uint32_t)k;
      s_eidx[lds_insert<2 * kAsmThreads>(s_etab, ea / (uint32_t)k, put)] = (uint8_t)at;
    }
    ne += total;
  }
  __syncthreads();
  // distinct nodes, ascending (at most kPlanNodes: one list at least names each)
  uint32_t mine[4] = {0, 0, 0, 0}, f = 0, nn;
  if(t < ne)
    for(int m = 0; m < k; ++m) {
      bool put;
      mine[m] = conn[(uint64_t)s_elem[t] * k + m];
      (void)lds_insert<2 * kPlanNodes>(s_ntab, mine[m], put);
      f |= put ? 1u << m : 0u;
    }
  uint32_t o = wg_scan((uint32_t)__popc(f), s_wave, t, nn);
  for(uint32_t j = t; j < kPlanNodes; j += kAsmThreads) s_uniq[j] = 0xffffffffu;
  __syncthreads();
  for(int m = 0; m < 4; ++m)
    if(f & (1u << m)) s_uniq[o++] = mine[m];
  __syncthreads();
  lds_sort<kPlanNodes>(s_uniq, t);
  uint32_t packed = 0;
  if(t < ne)
    for(int m = 0; m < k; ++m) packed |= lds_find(s_uniq, nn, mine[m]) << (8 * m);
  s_loc[t] = packed;
  for(uint32_t i = t; i < ninc; i += kAsmThreads) {
    const uint32_t ea = inc[i0 + i];
    bool put;
    s_inc[i] = (uint16_t)((uint32_t)s_eidx[lds_insert<2 * kAsmThreads>(s_etab, ea / (uint32_t)k, put)] << 2 |
                          ea % (uint32_t)k);
  }
  const uint32_t cb = contrib_ptr[blk0], nct = contrib_ptr[blk0 + nblk] - cb;
  for(uint32_t i = t; i < nct; i += kAsmThreads) s_contrib[i] = contrib[cb + i];
  __syncthreads();
  // block lists
  uint32_t nc = 0, ib = 0, cnt = 0, row = r0;
  const uint16_t* ctr = s_contrib;
  if(t < nblk) {
    uint32_t hi = r1;
    while(hi - row > 1) {
      const uint32_t mid = (row + hi) >> 1;
      if(row_ptr[mid] <= blk0 + t) row = mid; else hi = mid;
    }
    ib = inc_ptr[row];
    const uint32_t c0 = contrib_ptr[blk0 + t];
    ctr += c0 - cb;
    nc = contrib_ptr[blk0 + t + 1] - c0;
    for_block_lists(ctr, nc, periodic, k, len, inc + ib, conn, [&](auto, uint32_t) { ++cnt; });
  }
  uint32_t nlists;
  const uint32_t first = wg_scan(cnt, s_wave, t, nlists);
  if(t < 3) {
    // every workgroup's atomics on the same words would take longer than all the rest of the kernel: only
    // those that raise the maximum seen (a stale value costs an atomic, never a maximum)
    const uint32_t v = t == 0 ? nn : t == 1 ? ne : nlists;
    if(v > *static_cast<volatile const uint32_t*>(&most[t])) atomicMax(&most[t], v);
  }
  if(nn > ns) return;
  unsigned char* plan = plans + (uint64_t)wg * plan_bytes(ns);
  uint32_t* head = reinterpret_cast<uint32_t*>(plan);
  uint32_t* nodes = reinterpret_cast<uint32_t*>(plan + kPlanHeadBytes);
  uint32_t* loc = nodes + ns;
  uint64_t* lo = reinterpret_cast<uint64_t*>(loc + kAsmThreads);
  uint16_t* hi = reinterpret_cast<uint16_t*>(lo + kAsmThreads);
  if(t == 0) {
    head[0] = r0; head[1] = r1 - r0; head[2] = ne; head[3] = nn;
    head[4] = blk0; head[5] = nblk; head[6] = nlists; head[7] = 0;
  }
  for(uint32_t j = t; j < ns; j += kAsmThreads) nodes[j] = s_uniq[min(j, nn - 1)];
  loc[t] = packed;
  if(t < nblk) {
    uint32_t at = first;
    bool blk_first = true;
    const bool row_first = blk0 + t == row_ptr[row];
    const uint16_t* binc = s_inc + (ib - i0);
    for_block_lists(ctr, nc, periodic, k, len, inc + ib, conn, [&](auto pos, uint32_t n) {
      uint64_t w = blk_first ? 1ull << 63 : 0;
      uint32_t h = blk_first && row_first ? 0x8000u : 0;
#pragma unroll
      for(uint32_t m = 0; m < 6; ++m) {
        uint32_t entry = ne << 4;
        if(m < n) {
          const uint32_t c = ctr[pos(m)], b = c & 15u, ea = binc[c >> 4];
          entry = ea << 2 | b;
          if(m == 0) w |= (uint64_t)((s_loc[ea >> 2] >> (8 * b)) & 255u) << 55;
        }
        if(m < 5) w |= (uint64_t)entry << (11 * m);
        else h |= entry;
      }
      lo[at] = w;
      hi[at] = (uint16_t)h;
      ++at;
      blk_first = false;
    });
  }
  for(uint32_t j = nlists + t; j < kAsmThreads; j += kAsmThreads) { lo[j] = 0; hi[j] = 0; }
}

// out[i] = map[in[i]]
__global__ void k_map_nodes(uint64_t n, const uint32_t* __restrict__ in, const uint32_t* __restrict__ map,
                            uint32_t* __restrict__ out)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) out[i] = map[in[i]];
}

template<typename KeyT>
void radix_sort(Context& c, DevBuf& in, DevBuf& out, uint64_t n, int end_bit)
{
  size_t temp_bytes = 0;
  HIP_OK(hipcub::DeviceRadixSort::SortKeys(nullptr, temp_bytes, in.as<KeyT>(), out.as<KeyT>(), (int64_t)n, 0, end_bit,
                                           c.stream));
  DevBuf temp;
  temp.alloc(&c, std::max<size_t>(temp_bytes, 16));
  HIP_OK(hipcub::DeviceRadixSort::SortKeys(temp.ptr, temp_bytes, in.as<KeyT>(), out.as<KeyT>(), (int64_t)n, 0, end_bit,
                                           c.stream));
}

}  // namespace

void build_graph_structures(Lss& L)
{
  Context& c = *L.ctx;
  L.diag_blk.alloc(&c, sizeof(uint32_t) * std::max<uint32_t>(L.n_nodes, 1));
  hipLaunchKernelGGL(k_diag_blocks, dim3(grid_for(L.n_nodes, 256)), dim3(256), 0, c.stream, L.n_nodes,
                     L.row_ptr.as<uint32_t>(), L.cols.as<uint32_t>(), L.diag_blk.as<uint32_t>());
  HIP_OK(hipGetLastError());
  std::vector<uint32_t> diag(L.n_nodes);
  HIP_OK(hipMemcpyAsync(diag.data(), L.diag_blk.ptr, sizeof(uint32_t) * L.n_nodes, hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipStreamSynchronize(c.stream));
  for(uint32_t i = 0; i < L.n_nodes; ++i)
    if(diag[i] == 0xffffffffu)
      CF3_THROW(CF3HIP_ERR_INVALID_ARG, "node graph row " + std::to_string(i) + " has no diagonal block");
}

void build_element_structures(Lss& L)
{
  Context& c = *L.ctx;
  const Mesh& M = *L.mesh;
  const uint64_t N = L.n_nodes, E = M.n_elems, k = M.k;   // N block rows
  const uint64_t npairs = E * k * k, nek = E * k;
  // rows and columns of the element nodes (the mesh nodes, or their block rows under periodic links);
  // the gathers of the kernels (and the nodes of the assembly plans) keep the mesh nodes of M.conn
  DevBuf dconn;
  const uint32_t* conn = M.conn.as<uint32_t>();
  if(L.periodic) {
    dconn.alloc(&c, sizeof(uint32_t) * nek);
    hipLaunchKernelGGL(k_map_nodes, dim3(grid_for(nek, 256)), dim3(256), 0, c.stream, nek, M.conn.as<uint32_t>(),
                       L.p2m.as<uint32_t>(), dconn.as<uint32_t>());
    HIP_OK(hipGetLastError());
    conn = dconn.as<uint32_t>();
  }

  // ---- node graph ----
  {
    DevBuf keys, sorted;
    keys.alloc(&c, sizeof(uint64_t) * npairs);
    sorted.alloc(&c, sizeof(uint64_t) * npairs);
    hipLaunchKernelGGL(k_pair_keys, dim3(grid_for(npairs, 256)), dim3(256), 0, c.stream, conn, (uint32_t)E, (int)k, N,
                       keys.as<uint64_t>());
    HIP_OK(hipGetLastError());
    radix_sort<uint64_t>(c, keys, sorted, npairs, bits_for(N * N - 1));
    // unique
    DevBuf nsel;
    nsel.alloc(&c, sizeof(int64_t));
    size_t temp_bytes = 0;
    HIP_OK(hipcub::DeviceSelect::Unique(nullptr, temp_bytes, sorted.as<uint64_t>(), keys.as<uint64_t>(),
                                        nsel.as<int64_t>(), (int64_t)npairs, c.stream));
    DevBuf temp;
    temp.alloc(&c, std::max<size_t>(temp_bytes, 16));
    HIP_OK(hipcub::DeviceSelect::Unique(temp.ptr, temp_bytes, sorted.as<uint64_t>(), keys.as<uint64_t>(),
                                        nsel.as<int64_t>(), (int64_t)npairs, c.stream));
    int64_t nb = 0;
    HIP_OK(hipMemcpyAsync(&nb, nsel.ptr, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
    HIP_OK(hipStreamSynchronize(c.stream));
    if(nb >= (int64_t)0xffffffffll)
      CF3_THROW(CF3HIP_ERR_LIMIT, "more than 2^32-1 node blocks");
    L.n_blocks = (uint64_t)nb;
    L.row_ptr.alloc(&c, sizeof(uint32_t) * (N + 1));
    L.cols.alloc(&c, sizeof(uint32_t) * std::max<uint64_t>(nb, 1));
    hipLaunchKernelGGL(k_row_ptr_from_keys, dim3(grid_for(N + 1, 256)), dim3(256), 0, c.stream, keys.as<uint64_t>(),
                       (uint64_t)nb, N, N, L.row_ptr.as<uint32_t>());
    hipLaunchKernelGGL(k_cols_from_keys, dim3(grid_for(nb, 256)), dim3(256), 0, c.stream, keys.as<uint64_t>(),
                       (uint64_t)nb, N, L.cols.as<uint32_t>());
    HIP_OK(hipGetLastError());
  }
  build_graph_structures(L);

  // ---- element-to-slot map ----
  L.slots.alloc(&c, sizeof(uint32_t) * npairs);
  hipLaunchKernelGGL(k_slots, dim3(grid_for(npairs, 256)), dim3(256), 0, c.stream, conn, (uint32_t)E, (int)k,
                     L.row_ptr.as<uint32_t>(), L.cols.as<uint32_t>(), L.slots.as<uint32_t>());
  HIP_OK(hipGetLastError());

  // ---- node -> (element, local node) incidences sorted by element ----
  L.inc_ptr.alloc(&c, sizeof(uint32_t) * (N + 1));
  L.inc.alloc(&c, sizeof(uint32_t) * nek);
  {
    DevBuf keys, sorted;
    keys.alloc(&c, sizeof(uint64_t) * nek);
    sorted.alloc(&c, sizeof(uint64_t) * nek);
    hipLaunchKernelGGL(k_inc_keys, dim3(grid_for(nek, 256)), dim3(256), 0, c.stream, conn, nek, keys.as<uint64_t>());
    HIP_OK(hipGetLastError());
    radix_sort<uint64_t>(c, keys, sorted, nek, bits_for(N * nek - 1));
    hipLaunchKernelGGL(k_row_ptr_from_keys, dim3(grid_for(N + 1, 256)), dim3(256), 0, c.stream,
                       sorted.as<uint64_t>(), nek, N, nek, L.inc_ptr.as<uint32_t>());
    hipLaunchKernelGGL(k_inc_from_keys, dim3(grid_for(nek, 256)), dim3(256), 0, c.stream, sorted.as<uint64_t>(), nek,
                       L.inc.as<uint32_t>());
    HIP_OK(hipGetLastError());
  }

  const bool q1 = is_cell(M.etype);   // one lane per column node (and Gauss point)
  const int lanes = cell_lanes(M.etype, (int)k);
  L.passes = q1 ? 1 : (int)k;
  L.pos_stride = q1 ? lanes : 4;

  // ---- per-slot contribution lists sorted by (slot, b, q) ----
  DevBuf contrib_ptr, contrib, acc_cnt, row_acc;
  contrib_ptr.alloc(&c, sizeof(uint32_t) * (L.n_blocks + 1));
  contrib.alloc(&c, sizeof(uint16_t) * npairs);
  {
    DevBuf keys, sorted;
    keys.alloc(&c, sizeof(uint64_t) * npairs);
    sorted.alloc(&c, sizeof(uint64_t) * npairs);
    hipLaunchKernelGGL(k_contrib_keys, dim3(grid_for(nek, 256)), dim3(256), 0, c.stream, conn, L.inc.as<uint32_t>(),
                       L.inc_ptr.as<uint32_t>(), L.slots.as<uint32_t>(), nek, (int)k, keys.as<uint64_t>());
    HIP_OK(hipGetLastError());
    radix_sort<uint64_t>(c, keys, sorted, npairs, bits_for(((uint64_t)L.n_blocks << 16) - 1));
    hipLaunchKernelGGL(k_row_ptr_from_keys, dim3(grid_for(L.n_blocks + 1, 256)), dim3(256), 0, c.stream,
                       sorted.as<uint64_t>(), npairs, L.n_blocks, (uint64_t)65536, contrib_ptr.as<uint32_t>());
    hipLaunchKernelGGL(k_contrib_from_keys, dim3(grid_for(npairs, 256)), dim3(256), 0, c.stream,
                       sorted.as<uint64_t>(), npairs, contrib.as<uint16_t>());
    HIP_OK(hipGetLastError());
  }
  // accumulator threads per block and per row
  // (block lists: the specialised simplex kernels, which take systems of dim + 1 equations only)
  const bool plans = !q1 && L.neq == M.dim + 1;
  const uint32_t list_len = plans ? plan_list_length((int)k) : 0;
  acc_cnt.alloc(&c, L.n_blocks);
  row_acc.alloc(&c, sizeof(uint32_t) * N);
  hipLaunchKernelGGL(k_block_acc, dim3(grid_for(L.n_blocks, 256)), dim3(256), 0, c.stream, L.n_blocks, L.passes,
                     contrib_ptr.as<uint32_t>(), contrib.as<uint16_t>(), acc_cnt.as<uint8_t>());
  hipLaunchKernelGGL(k_row_acc, dim3(grid_for(N, 256)), dim3(256), 0, c.stream, (uint32_t)N, L.row_ptr.as<uint32_t>(),
                     acc_cnt.as<uint8_t>(), list_len, L.periodic, (int)k, contrib_ptr.as<uint32_t>(),
                     contrib.as<uint16_t>(), L.inc_ptr.as<uint32_t>(), L.inc.as<uint32_t>(), M.conn.as<uint32_t>(),
                     row_acc.as<uint32_t>());
  HIP_OK(hipGetLastError());

  // ---- host-side schedule of rows into assembly workgroups (structure only) ----
  std::vector<uint32_t> inc_ptr(N + 1), racc(N);
  HIP_OK(hipMemcpyAsync(inc_ptr.data(), L.inc_ptr.ptr, sizeof(uint32_t) * (N + 1), hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipMemcpyAsync(racc.data(), row_acc.ptr, sizeof(uint32_t) * N, hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipStreamSynchronize(c.stream));
  // a workgroup holds at most inc_limit incidences (simplices: one incidence per thread; Q1 cells:
  // one (incidence, column node) pair per thread) and kAsmThreads accumulator threads
  const uint64_t inc_limit = q1 ? kAsmThreads / lanes : kAsmThreads;
  std::vector<uint32_t> wg;
  wg.push_back(0);
  uint32_t r = 0;
  while(r < N) {
    uint32_t r1 = r;
    uint64_t ninc = 0, nacc = 0;
    while(r1 < N) {
      const uint64_t di = inc_ptr[r1 + 1] - inc_ptr[r1];
      const uint64_t da = racc[r1] & 0xffffu;
      if(di > inc_limit || da > (uint64_t)kAsmThreads)
        CF3_THROW(CF3HIP_ERR_LIMIT, "node " + std::to_string(r1) + " has " + std::to_string(di) +
                                        " incident elements and needs " + std::to_string(da) +
                                        " accumulators: above the assembly workgroup limits of " +
                                        std::to_string(inc_limit) + " and " + std::to_string(kAsmThreads));
      if(ninc + di > inc_limit || nacc + da > (uint64_t)kAsmThreads || r1 - r >= (uint32_t)kAsmThreads)
        break;
      ninc += di;
      nacc += da;
      ++r1;
    }
    wg.push_back(r1);
    r = r1;
  }
  L.n_wg = (uint32_t)(wg.size() - 1);
  L.wg_rows.alloc(&c, sizeof(uint32_t) * wg.size());
  HIP_OK(hipMemcpyAsync(L.wg_rows.ptr, wg.data(), sizeof(uint32_t) * wg.size(), hipMemcpyHostToDevice, c.stream));

  // ---- staging maps ----
  L.inc_pos.alloc(&c, (size_t)nek * L.pos_stride);
  L.blk_beg.alloc(&c, (size_t)L.n_blocks * 4);
  L.blk_acc.alloc(&c, sizeof(uint16_t) * L.n_blocks);
  lss_fill8(c, L.inc_pos.as<uint8_t>(), (size_t)nek * L.pos_stride, 0);
  hipLaunchKernelGGL(k_stage_maps, dim3(L.n_wg), dim3(kAsmThreads), 0, c.stream, L.passes, L.pos_stride,
                     L.wg_rows.as<uint32_t>(), L.row_ptr.as<uint32_t>(), L.inc_ptr.as<uint32_t>(),
                     contrib_ptr.as<uint32_t>(), contrib.as<uint16_t>(), acc_cnt.as<uint8_t>(),
                     L.inc_pos.as<uint8_t>(), L.blk_beg.as<uint8_t>(), L.blk_acc.as<uint16_t>());
  HIP_OK(hipGetLastError());

  // ---- assembly plans (specialised simplices) ----
  if(plans && N > 0) {
    // one allocation: info (n_plan, misfit, most[3]), workgroup starts, start flags, back, room of the selection
    const hipcub::CountingInputIterator<uint32_t> rows(0);
    size_t temp_bytes = 0;
    HIP_OK(hipcub::DeviceSelect::Flagged(nullptr, temp_bytes, rows, (uint8_t*)nullptr, (uint32_t*)nullptr,
                                         (uint32_t*)nullptr, (int)N, c.stream));
    const size_t head = (32 + 5 * N + nek + 255) / 256 * 256;
    DevBuf scratch;
    scratch.alloc(&c, head + std::max<size_t>(temp_bytes, 16));
    uint32_t* inf = scratch.as<uint32_t>();
    uint32_t* starts = inf + 8;
    uint8_t* flag = reinterpret_cast<uint8_t*>(starts + N);
    uint8_t* back = flag + N;
    uint32_t host[5];
    hipLaunchKernelGGL(k_inc_back, dim3(grid_for(nek, 256)), dim3(256), 0, c.stream, nek, (int)k, L.inc.as<uint32_t>(),
                       conn, back, inf);
    hipLaunchKernelGGL(k_plan_partition, dim3(grid_for(N, plan_segment(N))), dim3(64), 0, c.stream, (uint32_t)N,
                       plan_segment(N), L.inc_ptr.as<uint32_t>(), back, row_acc.as<uint32_t>(), flag,
                       reinterpret_cast<int*>(inf + 1));
    HIP_OK(hipcub::DeviceSelect::Flagged(scratch.as<char>() + head, temp_bytes, rows, flag, starts, inf, (int)N,
                                         c.stream));
    HIP_OK(hipMemcpyAsync(host, inf, sizeof(host), hipMemcpyDeviceToHost, c.stream));
    HIP_OK(hipStreamSynchronize(c.stream));
    const uint32_t n_plan = host[0];
    // node slots: most meshes need few; a workgroup that needs more is counted, and the plans are made again
    for(uint32_t ns = 64; !host[1];) {
      L.plan.alloc(&c, (size_t)n_plan * plan_bytes(ns));
      hipLaunchKernelGGL(k_plan_fill, dim3(n_plan), dim3(kAsmThreads), 0, c.stream, (uint32_t)N, n_plan, (int)k, list_len,
                         L.periodic, ns, starts, L.row_ptr.as<uint32_t>(), L.inc_ptr.as<uint32_t>(),
                         L.inc.as<uint32_t>(), back, conn, M.conn.as<uint32_t>(),
                         contrib_ptr.as<uint32_t>(), contrib.as<uint16_t>(), L.plan.as<unsigned char>(), inf + 2);
      HIP_OK(hipGetLastError());
      HIP_OK(hipMemcpyAsync(host, inf, sizeof(host), hipMemcpyDeviceToHost, c.stream));
      HIP_OK(hipStreamSynchronize(c.stream));
      if(host[2] <= ns) {
        L.n_plan = n_plan;
        L.plan_nodes = ns;
        L.plan_elems = host[3];
        L.plan_lists = host[4];
        break;
      }
      L.plan.release();
      ns = (host[2] + 3) / 4 * 4;   // at most kPlanNodes
    }
  }
  HIP_OK(hipStreamSynchronize(c.stream));
}

}  // namespace cf3hip
