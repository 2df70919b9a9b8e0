// The outer RFC 6962 Merkle tree over leaf digests, on gfx950.
//
// Reference: verification/commitment/native.c:312-337 (build_tree, pots_merkle_tree) and
// verification/commitment/merkle.py:153-224 (hash_node, _split, merkle_root, _tree_nodes).
//
// The tree is written straight into the pre-order node buffer the reference defines: the node
// of a range [lo, hi) with n > 1 leaves sits at p, its left child (the first k leaves, k the
// largest power of two below n) at p + 1 and its right child at p + 2k. The tree is built level
// by level: at level l the ranges are [j 2^l, min((j + 1) 2^l, n)); a range that fits in one
// level-(l-1) range is the same node as that child (RFC 6962 promotes an unpaired node rather
// than duplicating it), so only ranges longer than 2^(l-1) are hashed. A block takes kTreeTile
// neighbouring nodes of one level through the eight levels above them in LDS, so a launch
// covers eight levels and 65536 leaves take two.
//
// H_node(l, r) = BLAKE3(0x01 || l || r): a 65-byte message, one chunk of two blocks.
#include <string.h>

#include "blake3_device.h"
#include "common.h"

namespace pots {

// The pre-order slot of the node over [lo, min(lo + 2^level, n)), lo a multiple of 2^level. On
// the way down from the root every right turn adds 2k, k the leaves it passes, and every left
// turn adds 1: the right turns sum to 2·lo. The way follows the right edge of the tree, whose
// ranges begin at the prefixes of n - 1's bits, as far as lo's bits agree with them; where they
// first differ (bit t, set in n - 1) it turns left into a full subtree of 2^t leaves, in which
// it turns right at each set bit of lo and left at the others, down to 2^level leaves.
__device__ __forceinline__ uint64_t preorder_slot(uint64_t lo, uint32_t level, uint64_t n) {
  const uint64_t differ = (lo ^ (n - 1)) >> level;
  if (differ == 0) return 2 * lo;  // on the right edge itself
  const uint32_t t = level + 63 - __clzll(differ);
  return 2 * lo + 1 + (t - level) - __popcll(lo & ((1ull << t) - 1));
}

__device__ __forceinline__ void load8(const uint8_t* p, uint32_t w[8]) {
  const uint4* q = reinterpret_cast<const uint4*>(p);
  const uint4 a = q[0], b = q[1];
  w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
  w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
}

__device__ __forceinline__ void store8(uint8_t* p, const uint32_t w[8]) {
  uint4* q = reinterpret_cast<uint4*>(p);
  q[0] = make_uint4(w[0], w[1], w[2], w[3]);
  q[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

constexpr uint32_t kTreeLevels = 8, kTreeTile = 1u << kTreeLevels;

// Nodes of one level, in pairs 20 words apart (a pair is the 64 bytes hashed after the 0x01).
__device__ __forceinline__ uint32_t node_at(uint32_t j) { return (j >> 1) * 20 + (j & 1) * 8; }

// Block b: nodes b·kTreeTile .. of level `base` (ranges of 2^base leaves), read from the leaves
// (base 0, which it also places in their slots) or from their slots, and the levels above them
// up to base + kTreeLevels. Each hash is two compressions in a row, so it is the latency of the
// levels that counts: four lanes share a compression (b3_quad_compress).
//
// (A launch per level, one lane per node, and a walk down from the root for each node's slot:
// 147, 677, 9335, 65536 and 1000000 leaves took 42, 53, 79, 94 and 173 us with the call's own
// 10; this takes 22, 28, 34, 40 and 113.)
__global__ __launch_bounds__(256) void tree_kernel(const uint8_t* __restrict__ leaves,
                                                   uint8_t* __restrict__ nodes, uint64_t n,
                                                   uint32_t base) {
  __shared__ __align__(16) uint32_t s_a[kTreeTile / 2 * 20], s_b[kTreeTile / 4 * 20];
  __shared__ __align__(16) uint32_t s_msg[64 * 36];  // a quad's message: two blocks
  const uint32_t tid = threadIdx.x, q = tid & 3, quad = tid >> 2;
  const uint64_t count = ((n - 1) >> base) + 1;
  const uint64_t first = (uint64_t)blockIdx.x * kTreeTile;
  uint32_t m = (uint32_t)min<uint64_t>(kTreeTile, count - first);
  if (tid < m) {
    const uint64_t lo = (first + tid) << base, slot = preorder_slot(lo, base, n);
    uint32_t w[8];
    load8(base == 0 ? leaves + 32 * lo : nodes + 32 * slot, w);
    store8(reinterpret_cast<uint8_t*>(s_a + node_at(tid)), w);
    if (base == 0) store8(nodes + 32 * slot, w);
  }
  const B3Quad sched = b3_quad_schedule(q);
  uint32_t* const msg = s_msg + 36 * quad;
  uint32_t *cur = s_a, *nxt = s_b;
  for (uint32_t level = base + 1; m > 1; level++) {
    __syncthreads();
    const uint64_t j0 = first >> (level - base);
    for (uint32_t t = quad; 2 * t < m; t += 64) {
      const uint32_t* s = cur + 20 * t;
      uint32_t* dst = nxt + node_at(t);
      if (2 * t + 1 == m) {  // promoted: the same node as its only child
        dst[q] = s[q];
        dst[4 + q] = s[4 + q];
        continue;
      }
      // 0x01 || l || r: the sixteen words moved up by a byte, the last byte in a block of its own
#pragma unroll
      for (uint32_t u = 0; u < 4; u++) {
        const uint32_t i = 4 * q + u;
        msg[i] = (i == 0 ? 0x01u : s[max(i, 1u) - 1] >> 24) | s[i] << 8;
        msg[16 + i] = i == 0 ? s[15] >> 24 : 0u;
      }
      wave_sync();  // a lane reads words that its quad's other lanes wrote
      uint32_t lo, hi;
      b3_quad_iv(q, lo, hi);
      b3_quad_compress(sched, msg, q, q == 2 ? 64u : q == 3 ? B3_CHUNK_START : 0u, lo, hi);
      b3_quad_compress(sched, msg + 16, q,
                       q == 2   ? 1u
                       : q == 3 ? (uint32_t)(B3_CHUNK_END | B3_ROOT)
                                : 0u,
                       lo, hi);
      wave_sync();  // the quad's next message goes where this one was read
      dst[q] = lo;
      dst[4 + q] = hi;
      uint32_t* node = reinterpret_cast<uint32_t*>(
          nodes + 32 * preorder_slot((j0 + t) << level, level, n));
      node[q] = lo;
      node[4 + q] = hi;
    }
    m = (m + 1) / 2;
    uint32_t* const swap = cur;
    cur = nxt;
    nxt = swap;
  }
}

static int tree_enqueue(size_t n, const uint8_t* d_leaves, uint8_t* d_nodes, hipStream_t s) {
  uint64_t count = n;
  for (uint32_t base = 0;; base += kTreeLevels) {
    const uint64_t blocks = (count + kTreeTile - 1) / kTreeTile;
    hipLaunchKernelGGL(tree_kernel, dim3((uint32_t)blocks), dim3(256), 0, s, d_leaves, d_nodes,
                       (uint64_t)n, base);
    POTS_HIP(hipGetLastError());
    if (blocks == 1) return POTS_E_OK;
    count = blocks;
  }
}

}  // namespace pots

using namespace pots;

extern "C" int pots_merkle_tree_async(size_t n, const uint8_t* d_leaves, uint8_t* d_nodes,
                                      void* stream) {
  if (n == 0 || !d_leaves || !d_nodes) return POTS_E_ARG;
  return tree_enqueue(n, d_leaves, d_nodes, static_cast<hipStream_t>(stream));
}

extern "C" int pots_merkle_tree(size_t n, const uint8_t* leaves, uint8_t* nodes) {
  if (n == 0 || !leaves || !nodes) return POTS_E_ARG;
  const bool dev_in = is_device_pointer(leaves), dev_out = is_device_pointer(nodes);
  const size_t in_bytes = 32 * n, out_bytes = 32 * (2 * n - 1);
  const uint8_t* d_in = leaves;
  uint8_t* d_out = nodes;
  int rc;
  if (!dev_in || !dev_out) {
    void* buf = nullptr;
    if ((rc = arena_get(2, align_up(in_bytes, 256) + out_bytes, &buf)) != POTS_E_OK) return rc;
    if (!dev_in) {
      POTS_HIP(hipMemcpy(buf, leaves, in_bytes, hipMemcpyHostToDevice));
      d_in = static_cast<const uint8_t*>(buf);
    }
    if (!dev_out) d_out = static_cast<uint8_t*>(buf) + align_up(in_bytes, 256);
  }
  if ((rc = tree_enqueue(n, d_in, d_out, 0)) != POTS_E_OK) return rc;
  if (!dev_out) POTS_HIP(hipMemcpy(nodes, d_out, out_bytes, hipMemcpyDeviceToHost));
  else POTS_HIP(hipDeviceSynchronize());
  return POTS_E_OK;
}
