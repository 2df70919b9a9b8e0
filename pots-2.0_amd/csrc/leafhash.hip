// Leaf hashing on gfx950: H_leaf = BLAKE3(0x00 || header || payload) for every leaf of a
// transcript in one pass over HBM, with the NaN/Inf test fused into the loads.
//
// Reference: verification/commitment/native.c:171-259 (pots_hash_leaves, hash_leaf,
// leaf_worker) and verification/commitment/leaves.py:312-437 (the batching around it).
//
// Decomposition. Every leaf's message is cut into BLAKE3's 1 KiB chunks; one lane (or, in a
// plan of few chunks, four) compresses one chunk (up to 16 blocks) and writes its chaining
// value, or the digest itself when the leaf is a single chunk. The chunk CVs of a leaf form
// BLAKE3's tree, which has the RFC 6962 shape (a run of n > 1 chunks splits at the largest
// power of two below n), so it is reduced level by level, ten levels a launch (three, where a plan
// holds many short leaves): level l+1 node j is the parent of level-l nodes 2j and 2j+1, or node
// 2j itself when it has no sibling. The node that covers the whole leaf gets the ROOT flag.
//
// Message layout in HBM. The 0x00 prefix and the tensor header are 4(1 + ndim) bytes, a whole
// number of words, so message word w of a leaf is payload word w - H/4 and no byte shifting is
// needed. A lane reads two 64-byte blocks at a time as 16-byte aligned loads and picks their
// 32 words out of the 36-word window with a shift SH (0..3) that is fixed per leaf; SH is a
// template parameter so the selection is register renaming. Blocks that touch the header, the end of
// the payload or a partial word take an edge path that patches header words in from a small
// table and masks bytes past the end. Leaves whose header length or payload address is not
// word aligned (records, odd views, host memory) are staged: their whole message is copied to
// an aligned device buffer first and hashed with an empty header.
//
// Finiteness. A value is NaN or Inf when its exponent field is all ones. Masking each payload
// word to its exponent fields and keeping a running per-16-bit-half maximum (one and, one
// packed max per word) reaches the all-ones pattern exactly when a non-finite value was seen.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <new>
#include <unordered_set>
#include <vector>

#include "blake3_device.h"
#include "common.h"
#include "freivalds.h"
#include "gmem.h"

namespace pots {

constexpr uint32_t kNoFuse = 0xFFFFFFFFu;

struct LeafDesc {
  uint64_t payload;    // device address of payload byte 0 (word aligned)
  uint64_t len;        // payload bytes
  uint32_t head_word;  // first word of this leaf's 0x00 || header in the head table
  uint32_t head_len;   // bytes of 0x00 || header, a multiple of 4 (0 for a staged leaf)
  uint32_t kind;       // POTS_KIND_*
  uint32_t fin_from;   // message byte where the payload (the NaN/Inf-tested bytes) begins
  uint64_t cv_first;   // where chunk 0's chaining value goes in the level-0 buffer
  uint32_t n_chunks;   // 1 KiB chunks of the message (at least 1)
  uint32_t fuse;       // index of its fused-product entry, or kNoFuse
};
static_assert(sizeof(LeafDesc) == 48, "LeafDesc layout");

// A leaf whose product's P-pass sums the chunk kernel takes (freivalds.h). Its first nf
// chunks are hashed in class order: class kappa = c mod T holds the chunks whose payload
// offset is the same modulo the row length. A lane hashes a run of consecutive chunks (of
// classes t0 .. t0 + RC − 1 of one period when T >= 4; of PG whole periods when T < 4), and
// the runs of one class range get Q lanes (Q a multiple of 64, padding lanes idle), so every
// wave is at one common column offset at each step of its runs: R is read with scalar loads,
// one copy for the wave. A last chunk with fewer than 128 bytes has no interior
// pair and no P-pass work; it is left out of the classes (nf = n_chunks - 1) and hashed by a
// wave of its own after them, so that the header's few bytes do not pad every class.
struct FuseDesc {
  uint64_t r;          // R [m][k] fp32, row-major
  uint64_t seg;        // run records [J][n_rows]
  uint32_t row_bytes;  // m · esz
  uint32_t n_rows;
  uint32_t J;          // record slots per row
  uint32_t T;          // classes
  uint32_t Q;          // lanes per class
  uint32_t esz;        // 2 (bf16) or 4 (fp32)
  uint32_t nf;         // chunks in class order
  uint32_t run;        // a lane's run: classes (low 16 bits) x periods (high 16 bits)
};
static_assert(sizeof(FuseDesc) == 48, "FuseDesc layout");

struct LevelEntry {     // one leaf with >= 2 nodes at the input level of one fold
  uint64_t in_off;      // its first node in the level's input buffer
  uint64_t out_off;     // its first node in the fold's output buffer
  uint64_t out_first;   // its first output, counted over the fold's entries
  uint32_t n_in;        // its nodes at this level
  uint32_t leaf;
};
static_assert(sizeof(LevelEntry) == 32, "LevelEntry layout");

constexpr int kThreads = 256;
// Consecutive chunks one lane hashes in a row, at most: each chunk after the first takes its
// first bytes from the unit its predecessor's last pair loaded, so the 128-byte line before a
// 1 KiB boundary is read once, not again by the next chunk.
constexpr uint32_t kRun = 4;
// Chunks per wave of the four-lane chunk kernel, and the words of one chunk's place in its LDS
// (1 KiB and 16 bytes: neighbouring quads' words sit 4 banks apart).
constexpr uint32_t kQuadChunks = 16, kQuadStride = 260;
// Tree levels one launch of level_kernel reduces, and the nodes a block takes to reduce them.
constexpr uint32_t kFold = 10, kTile = 1u << kFold;
// The same of level_lanes, of which a lane takes the nodes.
constexpr uint32_t kLaneFold = 3, kLaneTile = 1u << kLaneFold;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4w __attribute__((ext_vector_type(4), aligned(4)));  // word aligned
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The NaN/Inf test of a chunk's payload words, one accumulator per lane: `mask` keeps each
// value's exponent field (fp32 0x7F800000, bf16 0x7F807F80, fp16 0x7C007C00, none 0), and the
// running per-half maximum of the masked words reaches the all-ones exponent (0x7F80 for fp32
// and bf16, 0x7C00 for fp16) exactly when a non-finite value was seen. Two VALU operations per
// word (and, packed 16-bit max). (A per-kind test with one v_dot2c_f32_bf16 per word measured
// slower: the chunk kernel's code doubles and its time went up by 5%.)
struct Fin {
  u16x2 acc = {0, 0};
  uint32_t mask;
  unsigned short thr;
  __device__ __forceinline__ explicit Fin(uint32_t kind)
      : mask(kind == POTS_KIND_F32    ? 0x7F800000u
             : kind == POTS_KIND_BF16 ? 0x7F807F80u
             : kind == POTS_KIND_F16  ? 0x7C007C00u
                                      : 0u),
        thr(kind == POTS_KIND_F16 ? 0x7C00 : 0x7F80) {}
  __device__ __forceinline__ void add(uint32_t w) {
    acc = __builtin_elementwise_max(acc, __builtin_bit_cast(u16x2, w & mask));
  }
  __device__ __forceinline__ bool bad() const {
    return mask != 0u && (acc.x >= thr || acc.y >= thr);
  }
};

// ---- P-pass sums of a fused product leaf ---------------------------------------------------
//
// A lane keeps one run at a time: Σ x·R[col][j] (j < 4) and Σ|x| in fp32 over the run, Σx² in
// fp32 over each 128-byte pair and in fp64 across pairs. A run ends where its row does (the
// row boundary is at the same offset in every lane of the wave, so the branch is uniform) and
// at the end of the chunk, and is written as one record.
//
// Σx² in fp32 is exact to rounding only while the squares are normal and their sum finite: a
// run with a pair whose largest biased exponent (from the NaN/Inf test's per-pair maximum) is
// outside [kSqLo, kSqHi] (|x| below 2^-50 or from 2^63 on) is marked in its record, and the
// P stage then takes that row's squares in fp64 from P, as the unfused P pass does.

constexpr uint32_t kSqLo = 127 - 50, kSqHi = 127 + 62;

typedef float v4f32 __attribute__((ext_vector_type(4)));
#define POTS_CONST __attribute__((address_space(4)))

struct PRun {
  float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f, s1 = 0.f;
  double s2 = 0.0;
  bool live = false;
  bool exact = false;  // a pair's exponents leave fp32 squares' range: the row is redone in fp64
};

// The elements t in [lo, hi) of a 128-byte pair (words w[0..31] of payload) into the run;
// element t's column is R row rcol + t (rcol: wave-uniform address of R's row for t = 0; a
// row is the plan's K challenges, K of 1, 2 or 4). Unmasked, every element of the pair is
// taken and the bounds are not read.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Elements t in [lo, hi) of a pair (its 32 payload words w) into the run. `emax`: the pair's
// largest biased exponent; outside [kSqLo, kSqHi] the run is marked for the exact squares.
typedef float v2f32 __attribute__((ext_vector_type(2)));

//
// `s1p`, `q2p`: an unmasked bf16 pair's Σ|x| and Σx², taken with the NaN/Inf test (unused
// otherwise). `zero`: every element of the pair is zero, whose squares are exact whatever the
// exponent test says.
template <int ESZ, bool MASKED, int K>
__device__ __forceinline__ void run_add(const uint32_t* w, float s1p, float q2p, uint64_t rcol,
                                        uint32_t lo, uint32_t hi, uint32_t emax, bool zero,
                                        PRun& a) {
  constexpr int NE = 128 / ESZ;
  static_assert(K == 1 || K == 2 || K == 4, "R rows of 1, 2 or 4 challenges");
  float q = 0.f;
#pragma unroll
  for (int t = 0; t < NE; t++) {
    if (MASKED && !((uint32_t)t >= lo && (uint32_t)t < hi)) continue;
    uint32_t wt = w[ESZ == 2 ? t >> 1 : t];
    // A masked pair is taken in two calls over the same words: an empty asm statement per
    // element keeps each conversion under its own bounds test, where the compiler would
    // otherwise convert all of the pair's elements once, ahead of both calls, and hold them.
    if (MASKED) asm volatile("" : "+v"(wt));
    float x;
    if (ESZ == 2) x = __uint_as_float((t & 1) ? (wt & 0xFFFF0000u) : (wt << 16));
    else x = __uint_as_float(wt);
    if constexpr (K == 4) {
      const v4f32 r = reinterpret_cast<const POTS_CONST v4f32*>(rcol)[t];
      a.d0 = fmaf(x, r[0], a.d0);
      a.d1 = fmaf(x, r[1], a.d1);
      a.d2 = fmaf(x, r[2], a.d2);
      a.d3 = fmaf(x, r[3], a.d3);
    } else if constexpr (K == 2) {
      const v2f32 r = reinterpret_cast<const POTS_CONST v2f32*>(rcol)[t];
      a.d0 = fmaf(x, r[0], a.d0);
      a.d1 = fmaf(x, r[1], a.d1);
    } else {
      a.d0 = fmaf(x, reinterpret_cast<const POTS_CONST float*>(rcol)[t], a.d0);
    }
    if (MASKED || ESZ == 4) {
      a.s1 += fabsf(x);
      q = fmaf(x, x, q);
    }
  }
  if (!MASKED && ESZ == 2) {
    a.s1 += s1p;
    q = q2p;
  }
  a.s2 += (double)q;
  a.exact |= (emax < kSqLo && !zero) || emax > kSqHi;
  a.live = true;
}

// Write the run of `row` in chunk c (message offset of the payload H) as its record: slot
// c − (chunk of the row's first element a chunk takes). Out-of-range indices are not written.
__device__ __forceinline__ void run_flush(const FuseDesc& f, uint64_t H, uint32_t row,
                                          uint64_t c, PRun& a) {
  if (a.live) {
    const uint64_t hc = (H + 127) & ~uint64_t(127);
    const uint64_t fs = max<uint64_t>(H + (uint64_t)row * f.row_bytes, hc);
    const uint64_t slot = c - (fs >> 10);
    if (row < f.n_rows && slot < f.J) {
      char* rec = reinterpret_cast<char*>(f.seg) +
                  (uint64_t)kRunBytes * (slot * f.n_rows + row);
      gstore<v4f32>(rec, v4f32{a.d0, a.d1, a.d2, a.d3});
      const uint64_t sb = (uint64_t)__double_as_longlong(a.s2);
      gstore<u32x4>(rec + 16, u32x4{__float_as_uint(a.s1), a.exact ? 1u : 0u, (uint32_t)sb,
                                    (uint32_t)(sb >> 32)});
    }
  }
  a = PRun();
}

// Message block b of chunk c for the general case: blocks that touch the header, the end of
// the payload or a partial word. Header words come from the head table (a staged leaf holds
// its header in the staged message instead); bytes past the end are zero; only payload words
// (from fin_from on) feed the NaN/Inf test.
template <int SH>
__device__ __forceinline__ void edge_block(const LeafDesc& d, const uint32_t* __restrict__ head,
                                           uint64_t o, uint32_t m[16], Fin& fin) {
  const uint64_t H = d.head_len, L = H + d.len;
  const uint64_t pbeg = d.payload, pend = d.payload + d.len;
  const uint64_t A = d.payload + o - H;  // address of message byte o, in payload terms
  const u32x4* A16 = reinterpret_cast<const u32x4*>(A & ~uint64_t(15));
  uint32_t w[20];
#pragma unroll
  for (int u = 0; u < 5; u++) {
    const uint64_t X = reinterpret_cast<uint64_t>(A16 + u);
    u32x4 q = u32x4{0, 0, 0, 0};
    if ((u < 4 || SH) && X + 16 > pbeg && X < pend) q = gload<u32x4>(A16 + u);
    w[4 * u] = q.x;
    w[4 * u + 1] = q.y;
    w[4 * u + 2] = q.z;
    w[4 * u + 3] = q.w;
  }
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const uint64_t at = o + 4u * j;  // message byte offset of this word
    uint32_t mw = w[j + SH];
    if (at < H) {
      mw = gload<uint32_t>(head + d.head_word + (uint32_t)(at >> 2));
    } else if (at >= L) {
      mw = 0;
    } else {
      const uint64_t rem = L - at;
      if (rem < 4) mw &= (1u << (8 * rem)) - 1u;
      if (at >= d.fin_from) fin.add(mw);
    }
    m[j] = mw;
  }
}

// One lane's chunk c of leaf d: its chaining value (or the leaf digest when `root`). Blocks
// go in pairs: a pair wholly inside the payload is read as one 144-byte aligned window (nine
// 16-byte loads), so each 128-byte line a lane touches is used up by one group of loads
// instead of being fetched again for the second half; other pairs take edge_block.
//
// ESZ != 0 (a fused product leaf, SH == 1): each interior pair's elements also go into the
// lane's P-pass run.
//
// `carry`, `have_carry`: with SH != 0, the last unit the previous pair loaded, kept across the
// chunks of a lane's run (the caller starts a run with have_carry false; chunk c + 1's first
// window begins with chunk c's last unit).
template <int SH, int ESZ, int K = 4>
__device__ __forceinline__ void hash_chunk(const LeafDesc& d, const uint32_t* __restrict__ head,
                                           uint64_t c, bool root, uint32_t cv[8], Fin& fin,
                                           const FuseDesc& f, u32x4& carry, bool& have_carry) {
  const uint64_t H = d.head_len;
  const uint64_t L = H + d.len;
  const uint64_t cstart = c * 1024u;
  const uint64_t cbytes = min<uint64_t>(1024u, L - cstart);
  uint32_t nb = (uint32_t)((cbytes + 63) / 64);
  if (nb == 0) nb = 1;  // the empty message: one empty block
  b3_iv(cv);
  // With SH != 0 a pair's window starts with the last 16 bytes of the previous pair's line;
  // they are carried over in registers rather than loaded again (a second load of a line
  // already streamed past is often an HBM refetch).
  PRun run;
  uint32_t prow = 0, prb = 0;  // row of the next pair and its byte offset in the row
  bool pinit = false;
#pragma unroll 1
  for (uint32_t b = 0; b < nb; b += 2) {
    const uint64_t o = cstart + 64u * b;
    uint32_t m0[16], m1[16];
    if (o >= d.fin_from && o + 128 <= L) {
      const u32x4* A16 =
          reinterpret_cast<const u32x4*>((d.payload + o - H) & ~uint64_t(15));
      u32x4 q[9];
      if (SH) {
        if (have_carry) q[0] = carry;
        else q[0] = gload<u32x4>(A16);
#pragma unroll
        for (int u = 1; u < 9; u++) q[u] = gload<u32x4>(A16 + u);
        carry = q[8];
        have_carry = true;
      } else {
#pragma unroll
        for (int u = 0; u < 8; u++) q[u] = gload<u32x4>(A16 + u);
        q[8] = u32x4{0, 0, 0, 0};
      }
      uint32_t w[36];
#pragma unroll
      for (int u = 0; u < 9; u++) {
        w[4 * u] = q[u].x;
        w[4 * u + 1] = q[u].y;
        w[4 * u + 2] = q[u].z;
        w[4 * u + 3] = q[u].w;
      }
#pragma unroll
      for (int j = 0; j < 16; j++) {
        m0[j] = w[j + SH];
        m1[j] = w[16 + j + SH];
      }
      // The NaN/Inf test's per-pair maximum (a tree, then one merge into the running one). A
      // fused bf16 leaf's words are masked to |x| (sign bits cleared) instead of to their
      // exponents: a half reaches 0x7F80 for the same values, and the pair's Σ|x| takes the
      // masked words two elements per v_dot2 against (1, 1), beside Σx² from each word
      // against itself (products of bf16 values are exact in fp32).
      const uint32_t pmask = ESZ == 2 ? 0x7FFF7FFFu : fin.mask;
      u16x2 pm[8];
      float s1p = 0.f, q2p = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        uint32_t aw[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t wu = w[4 * j + e + SH];
          aw[e] = wu & pmask;
          if constexpr (ESZ == 2) {
            s1p = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, aw[e]),
                                                  __builtin_bit_cast(bf16x2, 0x3F803F80u), s1p,
                                                  false);
            q2p = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, wu),
                                                  __builtin_bit_cast(bf16x2, wu), q2p, false);
          }
        }
        pm[j] = __builtin_elementwise_max(
            __builtin_elementwise_max(__builtin_bit_cast(u16x2, aw[0]),
                                      __builtin_bit_cast(u16x2, aw[1])),
            __builtin_elementwise_max(__builtin_bit_cast(u16x2, aw[2]),
                                      __builtin_bit_cast(u16x2, aw[3])));
      }
#pragma unroll
      for (int j = 0; j < 4; j++) pm[j] = __builtin_elementwise_max(pm[j], pm[j + 4]);
      pm[0] = __builtin_elementwise_max(__builtin_elementwise_max(pm[0], pm[1]),
                                        __builtin_elementwise_max(pm[2], pm[3]));
      fin.acc = __builtin_elementwise_max(fin.acc, pm[0]);
      if constexpr (ESZ != 0) {
        // the pair's largest biased exponent: bf16 halves hold it at bit 7, fp32 at bit 23
        const uint32_t pmax = ESZ == 2 ? (uint32_t)max(pm[0].x, pm[0].y) : (uint32_t)pm[0].y;
        const uint32_t emax = pmax >> 7;
        // an all-zero pair, whose squares are exact (bf16; fp32's test keeps only exponents,
        // which do not tell zeros from subnormals)
        const bool zero = ESZ == 2 && pmax == 0;
        if (!pinit) {  // the chunk's first interior pair
          const uint64_t po = o - H;
          prow = (uint32_t)(po / f.row_bytes);
          prb = (uint32_t)(po - (uint64_t)prow * f.row_bytes);
          pinit = true;
        }
        // Every active lane holds the same offset (the class order), so these are scalars.
        // (readfirstlane returns int: each word goes through uint32_t before widening.)
        const uint32_t rb = (uint32_t)__builtin_amdgcn_readfirstlane(prb);
        const uint64_t rbase =
            (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(f.r >> 32)) << 32 |
            (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)f.r);
        if (rb + 128 <= f.row_bytes) {
          run_add<ESZ, false, K>(w + SH, s1p, q2p, rbase + (uint64_t)(rb / ESZ) * (4 * K), 0,
                                 128 / ESZ, emax, zero, run);
          prb = rb + 128;
          if (prb == f.row_bytes) {
            run_flush(f, H, prow, c, run);
            prow++;
            prb = 0;
          }
        } else {  // the pair ends row prow at element tb and starts row prow + 1
          const uint32_t tb = (f.row_bytes - rb) / ESZ;
          run_add<ESZ, true, K>(w + SH, 0.f, 0.f, rbase + (uint64_t)(rb / ESZ) * (4 * K), 0,
                                tb, emax, zero, run);
          run_flush(f, H, prow, c, run);
          prow++;
          run_add<ESZ, true, K>(w + SH, 0.f, 0.f, rbase - (uint64_t)tb * (4 * K), tb,
                                128 / ESZ, emax, zero, run);
          prb = rb + 128 - f.row_bytes;
        }
      }
      // Two whole 64-byte blocks of which the first never ends the chunk: the block lengths
      // are constant, and the chunk counter fits 32 bits (plan creation refuses a leaf of
      // 4 TiB or more).
      b3_compress_cv32(cv, m0, (uint32_t)c, 64u, b == 0 ? B3_CHUNK_START : 0u, cv);
      b3_compress_cv32(cv, m1, (uint32_t)c, 64u,
                       b + 2 == nb ? (B3_CHUNK_END | (root ? B3_ROOT : 0u)) : 0u, cv);
      continue;
    }
    edge_block<SH>(d, head, o, m0, fin);
    if (b + 1 < nb) edge_block<SH>(d, head, o + 64, m1, fin);
    have_carry = false;
    const uint32_t blen0 = (uint32_t)min<uint64_t>(64u, L > o ? L - o : 0u);
    uint32_t f0 = b == 0 ? B3_CHUNK_START : 0u;
    if (b + 1 == nb) f0 |= B3_CHUNK_END | (root ? B3_ROOT : 0u);
    b3_compress_cv(cv, m0, c, blen0, f0, cv);
    if (b + 1 < nb) {
      const uint32_t blen1 = (uint32_t)min<uint64_t>(64u, L - o - 64);
      const uint32_t f1 = b + 2 == nb ? (B3_CHUNK_END | (root ? B3_ROOT : 0u)) : 0u;
      b3_compress_cv(cv, m1, c, blen1, f1, cv);
    }
  }
  if constexpr (ESZ != 0) run_flush(f, H, prow, c, run);
}

// A chunk order: entry e covers slots first[e] .. first[e + 1] of leaf leaf[e], and the
// entries of block b's slots (kThreads of them; kQuadChunks for the four-lane kernel) lie in
// blk_ent[b] .. blk_ent[b + 1].
struct Order {
  const uint64_t* __restrict__ first;
  const uint32_t* __restrict__ leaf;
  const uint32_t* __restrict__ blk_ent;
  uint64_t n_slots;   // slots of the order
  uint32_t n_blocks;  // ceil(n_slots / slots per block)
  uint32_t run;       // chunks per slot (the plain order: lane_run)
  uint32_t short_most;
};

// Chunks per slot of a leaf of n chunks, in a plain order of runs of `run`: a leaf of up to
// short_most chunks takes runs of kRun, where those leave no more than 1/16 of their chunks empty
// (a leaf of up to kRun chunks is one run, whatever its length).
__host__ __device__ constexpr uint32_t lane_run(uint32_t n, uint32_t run, uint32_t short_most) {
  return n <= short_most && (n <= kRun || (kRun - 1 - (n + kRun - 1) % kRun) * 16 <= n) ? kRun
                                                                                        : run;
}

__device__ __forceinline__ uint32_t order_entry(const Order& od, uint64_t g, uint32_t blk) {
  uint32_t lo = od.blk_ent[blk], hi = od.blk_ent[blk + 1];
  while (lo < hi) {  // the last entry whose first slot is <= g
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (od.first[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ void store_cv(uint32_t* p, const uint32_t cv[8]) {
  u32x4* dst = reinterpret_cast<u32x4*>(p);
  gstore<u32x4>(dst, u32x4{cv[0], cv[1], cv[2], cv[3]});
  gstore<u32x4>(dst + 1, u32x4{cv[4], cv[5], cv[6], cv[7]});
}

// Chunks c0 .. c1 − 1 of leaf i, one after another on one lane, each chaining value to cv_out
// (or the leaf digest itself for a one-chunk leaf).
template <int SH>
__device__ __forceinline__ void hash_run(const LeafDesc& d, const uint32_t* __restrict__ head,
                                         uint32_t i, uint64_t c0, uint64_t c1, Fin& fin,
                                         uint32_t* __restrict__ cv_out,
                                         uint32_t* __restrict__ digests) {
  const FuseDesc none{};
  const bool root = d.n_chunks == 1;
  u32x4 carry = u32x4{0, 0, 0, 0};
  bool have_carry = false;
#pragma unroll 1
  for (uint64_t c = c0; c < c1; c++) {
    uint32_t cv[8];
    hash_chunk<SH, 0>(d, head, c, root, cv, fin, none, carry, have_carry);
    store_cv(root ? digests + 8ull * i : cv_out + 8ull * (d.cv_first + c), cv);
  }
}

// Every chunk of the unfused leaves: slot g of the plain order is run g − first[e] of leaf
// leaf[e], its chunks run·(g − first[e]) onwards, run the leaf's lane_run (slots past a leaf's runs
// are idle). Block b
// hashes slot blocks b, b + gridDim.x, ... so a grid smaller than the order holds a bounded
// share of the GPU and leaves the rest to kernels on other streams.
__global__ __launch_bounds__(kThreads) void chunk_kernel(
    const LeafDesc* __restrict__ leaves, Order od, const uint32_t* __restrict__ head,
    uint32_t* __restrict__ cv_out, uint32_t* __restrict__ digests,
    uint32_t* __restrict__ first_bad) {
  for (uint32_t blk = blockIdx.x; blk < od.n_blocks; blk += gridDim.x) {
    const uint64_t g = (uint64_t)blk * kThreads + threadIdx.x;
    if (g >= od.n_slots) continue;
    const uint32_t e = order_entry(od, g, blk);
    const uint32_t i = od.leaf[e];
    const LeafDesc d = leaves[i];
    const uint32_t run = lane_run(d.n_chunks, od.run, od.short_most);
    const uint64_t c0 = (g - od.first[e]) * run;
    if (c0 >= d.n_chunks) continue;
    const uint64_t c1 = min<uint64_t>(c0 + run, d.n_chunks);
    Fin fin(d.kind);
    switch ((uint32_t)((d.payload - d.head_len) >> 2) & 3u) {
      case 0: hash_run<0>(d, head, i, c0, c1, fin, cv_out, digests); break;
      case 1: hash_run<1>(d, head, i, c0, c1, fin, cv_out, digests); break;
      case 2: hash_run<2>(d, head, i, c0, c1, fin, cv_out, digests); break;
      default: hash_run<3>(d, head, i, c0, c1, fin, cv_out, digests); break;
    }
    if (fin.bad()) atomicMin(first_bad, i);
  }
}

// The chunks of the unfused leaves on four lanes each (b3_quad_compress), for plans of few
// chunks, where a chunk's sixteen serial compressions are the call's latency and most of the
// GPU would idle. A wave hashes kQuadChunks chunks. The quad's lanes load the chunk's sixteen
// blocks 16 bytes a lane, all in flight at once, into the wave's LDS: groups wholly inside the
// payload (past the header) as they lie, at word alignment, the loads of the others clamped
// into the payload and their words then rewritten one by one (header words, zeros past the
// end). No other wave touches that LDS, so a wave's own order, which it keeps by itself, is
// enough: wave_sync() only holds the compiler to it.
__global__ __launch_bounds__(64) void chunk_kernel_quad(
    const LeafDesc* __restrict__ leaves, Order od, const uint32_t* __restrict__ head,
    uint32_t* __restrict__ cv_out, uint32_t* __restrict__ digests,
    uint32_t* __restrict__ first_bad) {
  __shared__ __align__(16) uint32_t s_msg[kQuadChunks * kQuadStride];
  const uint32_t q = threadIdx.x & 3, slot = threadIdx.x >> 2;
  uint32_t* const msg = s_msg + slot * kQuadStride;
  const B3Quad sched = b3_quad_schedule(q);
  for (uint32_t blk = blockIdx.x; blk < od.n_blocks; blk += gridDim.x) {
    const uint64_t g = (uint64_t)blk * kQuadChunks + slot;
    if (g >= od.n_slots) continue;
    const uint32_t e = order_entry(od, g, blk);
    const uint32_t i = od.leaf[e];
    const LeafDesc d = leaves[i];
    const uint64_t c = g - od.first[e];  // < n_chunks: a slot per chunk
    const uint64_t H = d.head_len, L = H + d.len, cstart = c * 1024u;
    const uint64_t from = max<uint64_t>(H, d.fin_from);  // payload words begin here
    const uint64_t cbytes = min<uint64_t>(1024u, L - cstart);
    const uint32_t nb = max(1u, (uint32_t)((cbytes + 63) / 64));
    Fin fin(d.kind);
    if (d.len >= 16) {
      const uint64_t last = (d.len - 16) & ~uint64_t(3);
      u32x4 w[16];
#pragma unroll
      for (uint32_t b = 0; b < 16; b++) {
        const uint64_t o = cstart + 64u * b + 16u * q;
        w[b] = gload<u32x4w>(reinterpret_cast<const char*>(d.payload) +
                             (o < H ? 0 : min<uint64_t>(o - H, last)));
      }
#pragma unroll
      for (uint32_t b = 0; b < 16; b++) {
        const uint64_t o = cstart + 64u * b + 16u * q;
        if (o >= from && o + 16 <= L)
#pragma unroll
          for (int t = 0; t < 4; t++) fin.add(w[b][t]);
        *reinterpret_cast<u32x4*>(msg + 16 * b + 4 * q) = w[b];
      }
    }
    if (cstart < from || cstart + 1024 > L || d.len < 16) {
      for (uint32_t b = 0; b < nb; b++) {
        const uint64_t o = cstart + 64u * b + 16u * q;
        if (o >= from && o + 16 <= L && d.len >= 16) continue;
#pragma unroll
        for (uint32_t t = 0; t < 4; t++) {
          const uint64_t at = o + 4u * t;
          uint32_t mw = 0;
          if (at < H) {
            mw = gload<uint32_t>(head + d.head_word + (uint32_t)(at >> 2));
          } else if (at < L) {
            mw = gload<uint32_t>(reinterpret_cast<const char*>(d.payload) + (at - H));
            if (L - at < 4) mw &= (1u << (8 * (uint32_t)(L - at))) - 1u;
            if (at >= d.fin_from) fin.add(mw);
          }
          msg[16 * b + 4 * q + t] = mw;
        }
      }
    }
    wave_sync();
    const bool root = d.n_chunks == 1;
    uint32_t lo, hi;
    b3_quad_iv(q, lo, hi);
#pragma unroll 1
    for (uint32_t b = 0; b < nb; b++) {
      const uint32_t blen = min<uint32_t>(64u, (uint32_t)cbytes - 64u * b);
      uint32_t flags = b == 0 ? B3_CHUNK_START : 0u;
      if (b + 1 == nb) flags |= B3_CHUNK_END | (root ? B3_ROOT : 0u);
      const uint32_t tail = q == 0 ? (uint32_t)c : q == 1 ? 0u : q == 2 ? blen : flags;
      b3_quad_compress(sched, msg + 16 * b, q, tail, lo, hi);
    }
    uint32_t* out = root ? digests + 8ull * i : cv_out + 8ull * (d.cv_first + c);
    gstore<uint32_t>(out + q, lo);
    gstore<uint32_t>(out + 4 + q, hi);
    if (fin.bad()) atomicMin(first_bad, i);
    wave_sync();  // the next chunk's words go where these were read
  }
}

// With a block per order block, block b takes order block xcd_block(b, n) (gmem.h): each XCD
// hashes a contiguous range of the fused order, and neighbouring slots read the same rows of
// R, which one L2 then holds (the kernel's reads went from 1.12x to 1.05x its message bytes).
// The plain order has no R and keeps the hardware's interleave.
//
// The fused leaves (FuseDesc), each starting at a multiple of 64 slots in the fused order and
// holding a multiple of 64: a wave's slots are one leaf's and one class range's, so the entry,
// the leaf's descriptors and, at each step of the runs, R's rows are wave-uniform and live in
// scalar registers. Local slot l < NR·Q (NR = ceil(T / RC) class ranges) is the run of class
// range l / Q in period group l mod Q: chunks t0 + T·PG·(l mod Q) onwards (t0 = RC·(l / Q)),
// RC·PG of them, which are consecutive; the short last chunk follows.
template <int K>
__global__ __launch_bounds__(kThreads) void chunk_kernel_fused(
    const LeafDesc* __restrict__ leaves, const FuseDesc* __restrict__ fuses, Order od,
    const uint32_t* __restrict__ head, uint32_t* __restrict__ cv_out,
    uint32_t* __restrict__ first_bad) {
  const uint32_t wave_lane0 = threadIdx.x & ~63u;
  for (uint32_t b = blockIdx.x; b < od.n_blocks; b += gridDim.x) {
    const uint32_t blk = gridDim.x >= od.n_blocks ? xcd_block(b, od.n_blocks) : b;
    const uint64_t g0 = (uint64_t)blk * kThreads + wave_lane0;  // the wave's first slot
    if (g0 >= od.n_slots) continue;  // n_slots is a multiple of 64: whole waves
    const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane(order_entry(od, g0, blk));
    const uint32_t i = od.leaf[e];
    const LeafDesc d = leaves[i];
    const FuseDesc f = fuses[d.fuse];
    const uint32_t rc = f.run & 0xFFFFu, pg = f.run >> 16;
    const uint32_t tq = (f.T + rc - 1) / rc * f.Q;
    const uint32_t l32 = (uint32_t)(g0 - od.first[e]) + (threadIdx.x & 63u);  // < tq + 64
    Fin fin(d.kind);
    uint32_t cv[8];
    if (l32 < tq) {
      const uint32_t t0 = l32 / f.Q * rc;
      const uint64_t cs = (uint64_t)t0 + (uint64_t)f.T * pg * (l32 % f.Q);
      const uint64_t ce = min<uint64_t>(cs + (uint64_t)min(rc, f.T - t0) * pg, f.nf);
      u32x4 carry = u32x4{0, 0, 0, 0};
      bool have_carry = false;
#pragma unroll 1
      for (uint64_t c = cs; c < ce; c++) {
        if (f.esz == 2) hash_chunk<1, 2, K>(d, head, c, false, cv, fin, f, carry, have_carry);
        else hash_chunk<1, 4, K>(d, head, c, false, cv, fin, f, carry, have_carry);
        store_cv(cv_out + 8ull * (d.cv_first + c), cv);
      }
      if (cs >= ce) continue;
    } else {  // the short last chunk, if any
      const uint64_t c = (uint64_t)f.nf + (l32 - tq);
      if (c >= d.n_chunks) continue;
      u32x4 carry = u32x4{0, 0, 0, 0};
      bool have_carry = false;
      hash_chunk<1, 0>(d, head, c, false, cv, fin, f, carry, have_carry);
      store_cv(cv_out + 8ull * (d.cv_first + c), cv);
    }
    if (fin.bad()) atomicMin(first_bad, i);
  }
}

// Levels kFold at a time: block b makes one output node of its leaf (entry blk_ent[b]) at level
// l + kFold from the (at most kTile) nodes o·kTile .. of level l, with BLAKE3's rule at each
// level (pairs are hashed, a last odd node is promoted; kFold levels of it compose to a tile's
// own reduction, since tiles begin at multiples of kTile). A leaf whose tree closes inside the
// fold writes its digest: the compression that makes the single top node carries ROOT.
//
// A tile's first levels are wide, a lane per parent, the first straight from HBM; from 64
// parents on a level is one compression of latency on four lanes each (b3_quad_compress), the
// nodes in LDS throughout. (Three levels per launch, one lane each, took 44, 69, 80, 99 and
// 166 us for leaves of 1, 64, 256, 1024 and 4096 MiB; this takes 21, 27, 30, 54 and 132.)
//
// Node j lies at node_at(j): a pair is one 64-byte message, and pairs sit 20 words apart, so
// that the quads of a wave read different banks.
__device__ __forceinline__ uint32_t node_at(uint32_t j) { return (j >> 1) * 20 + (j & 1) * 8; }

__device__ __forceinline__ void lds_put8(uint32_t* p, const uint32_t v[8]) {
  *reinterpret_cast<u32x4*>(p) = u32x4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<u32x4*>(p + 4) = u32x4{v[4], v[5], v[6], v[7]};
}

__device__ __forceinline__ void get8(const u32x4& a, const u32x4& b, uint32_t v[8]) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    v[t] = a[t];
    v[4 + t] = b[t];
  }
}

__global__ __launch_bounds__(kThreads) void level_kernel(
    const LevelEntry* __restrict__ ents, const uint32_t* __restrict__ blk_ent,
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
    uint32_t* __restrict__ digests) {
  __shared__ __align__(16) uint32_t s_wide[kTile / 4 * 20];  // up to kTile / 2 nodes
  __shared__ __align__(16) uint32_t s_quad[32 * 20];         // up to 64 nodes
  const uint32_t tid = threadIdx.x;
  const LevelEntry e = ents[blk_ent[blockIdx.x]];
  const uint64_t o = blockIdx.x - e.out_first, first = o * kTile;
  const uint32_t cnt = (uint32_t)min<uint64_t>(kTile, e.n_in - first);
  const u32x4* src = reinterpret_cast<const u32x4*>(in + 8ull * (e.in_off + first));
  // m: the tile's nodes at the current level; n: the leaf's
  uint32_t m = cnt, n = e.n_in;
  if (cnt <= 128) {
    if (tid < 2 * cnt)
      *reinterpret_cast<u32x4*>(s_wide + node_at(tid >> 1) + 4 * (tid & 1)) =
          gload<u32x4>(src + tid);
    __syncthreads();
  } else {
    static_assert(kTile == 4 * kThreads, "two parents per thread at the first level");
    u32x4 x[2][4];
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
      const uint32_t t = tid + kThreads * h;
      // (a child past the tile rereads the tile's last node; its value is not used)
#pragma unroll
      for (uint32_t u = 0; u < 4; u++)
        x[h][u] = gload<u32x4>(src + 2 * min(2 * t + (u >> 1), cnt - 1) + (u & 1));
    }
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
      const uint32_t t = tid + kThreads * h;
      uint32_t l[8], r[8], v[8];
      get8(x[h][0], x[h][1], l);
      get8(x[h][2], x[h][3], r);
      if (2 * t + 1 < cnt) {
        b3_parent_cv(l, r, 0u, v);
        lds_put8(s_wide + node_at(t), v);
      } else if (2 * t < cnt) {
        lds_put8(s_wide + node_at(t), l);
      }
    }
    m = (m + 1) / 2;
    n = (n + 1) / 2;
    __syncthreads();
    while (m > 128) {
      uint32_t l[8], r[8], v[8];
      const bool pair = 2 * tid + 1 < m, one = 2 * tid < m;
      if (one) {
        const u32x4* p = reinterpret_cast<const u32x4*>(s_wide + 20 * tid);
        get8(p[0], p[1], l);
        get8(p[2], p[3], r);
      }
      __syncthreads();  // every child is read before a parent overwrites one
      if (pair) {
        b3_parent_cv(l, r, 0u, v);
        lds_put8(s_wide + node_at(tid), v);
      } else if (one) {
        lds_put8(s_wide + node_at(tid), l);
      }
      m = (m + 1) / 2;
      n = (n + 1) / 2;
      __syncthreads();
    }
  }
  const uint32_t q = tid & 3, t = tid >> 2;
  const B3Quad sched = b3_quad_schedule(q);
  uint32_t *cur = s_wide, *nxt = s_quad;
  while (m > 1) {
    n = (n + 1) / 2;
    const uint32_t flags = B3_PARENT | (n == 1 ? B3_ROOT : 0u);
    const uint32_t tail = q < 2 ? 0u : q == 2 ? 64u : flags;
    uint32_t* dst = nxt + node_at(t);
    if (2 * t + 1 < m) {
      uint32_t lo, hi;
      b3_quad_iv(q, lo, hi);
      b3_quad_compress(sched, cur + 20 * t, q, tail, lo, hi);
      dst[q] = lo;
      dst[4 + q] = hi;
    } else if (2 * t < m) {
      dst[q] = cur[20 * t + q];
      dst[4 + q] = cur[20 * t + 4 + q];
    }
    m = (m + 1) / 2;
    __syncthreads();
    uint32_t* const swap = cur;
    cur = nxt;
    nxt = swap;
  }
  if (tid < 8)
    gstore<uint32_t>((e.n_in <= kTile ? digests + 8ull * e.leaf : out + 8ull * (e.out_off + o)) +
                         tid,
                     cur[tid]);
}

// Levels kLaneFold at a time, for many short leaves (kShortLeast): lane t makes output t of the
// fold, node o of its leaf at level l + kLaneFold, from the (at most kLaneTile) nodes o·kLaneTile ..
// of level l, level by level in registers. The outputs of block b's lanes lie in entries blk_ent[b]
// .. blk_ent[b + 1]. Latency: seven compressions in a row and a search for the leaf, some 12 us a
// launch up to half a million nodes.
__global__ __launch_bounds__(kThreads) void level_lanes(
    const LevelEntry* __restrict__ ents, const uint32_t* __restrict__ blk_ent, uint64_t n_out,
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
    uint32_t* __restrict__ digests) {
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t >= n_out) return;
  uint32_t lo = blk_ent[blockIdx.x], hi = blk_ent[blockIdx.x + 1];
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (ents[mid].out_first <= t) lo = mid;
    else hi = mid - 1;
  }
  const LevelEntry e = ents[lo];
  const uint64_t o = t - e.out_first, first = o * kLaneTile;
  // m: the lane's nodes at the current level; n: the leaf's
  uint32_t m = (uint32_t)min<uint64_t>(kLaneTile, e.n_in - first), n = e.n_in;
  const u32x4* src = reinterpret_cast<const u32x4*>(in + 8ull * (e.in_off + first));
  uint32_t cv[kLaneTile][8];
#pragma unroll
  for (uint32_t a = 0; a < kLaneTile; a++) {
    u32x4 x = {0, 0, 0, 0}, y = {0, 0, 0, 0};
    if (a < m) {
      x = gload<u32x4>(src + 2 * a);
      y = gload<u32x4>(src + 2 * a + 1);
    }
    get8(x, y, cv[a]);
  }
#pragma unroll
  for (uint32_t lvl = 0; lvl < kLaneFold; lvl++) {
    n = (n + 1) / 2;
    const uint32_t flags = n == 1 ? B3_ROOT : 0u;
#pragma unroll
    for (uint32_t a = 0; a < (kLaneTile >> (lvl + 1)); a++) {
      if (2 * a + 1 < m) {
        b3_parent_cv(cv[2 * a], cv[2 * a + 1], flags, cv[a]);
      } else if (2 * a < m) {
#pragma unroll
        for (int q = 0; q < 8; q++) cv[a][q] = cv[2 * a][q];
      }
    }
    m = (m + 1) / 2;
  }
  store_cv(e.n_in <= kLaneTile ? digests + 8ull * e.leaf : out + 8ull * (e.out_off + o), cv[0]);
}

// Messages that are not word aligned where they lie (a record, a view at an odd element) are
// staged: 0x00 || header || payload in one aligned buffer. One launch writes them all, 16 bytes
// a thread, and resets the first-bad word; a payload in host memory (to == head) is copied in
// after it. (Two device copies per leaf and the reset, each a launch of its own, were 17 launches
// and about 80 us for eight records.)
struct StageJob {
  uint64_t payload;    // device address of the payload, at any alignment
  uint32_t leaf;       // whose descriptor holds where the message goes (16-byte aligned, with room
                       // to a multiple of 16 bytes), its bytes and those of its head
  uint32_t head_word;  // first word of the head bytes in the head table
  uint32_t blk_first;  // prefix of blocks over the jobs before it
  uint32_t host;       // the payload is in host memory: only the head is written
};
static_assert(sizeof(StageJob) == 24, "StageJob layout");
constexpr uint32_t kStageBytes = 16 * kThreads;  // of a message, per block

__global__ __launch_bounds__(kThreads) void stage_kernel(const StageJob* __restrict__ jobs,
                                                         uint32_t n_jobs,
                                                         const LeafDesc* __restrict__ leaves,
                                                         const uint32_t* __restrict__ head_table,
                                                         uint32_t* first_bad, uint32_t n_leaves) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *first_bad = n_leaves;
  if (n_jobs == 0) return;
  uint32_t lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (jobs[mid].blk_first <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const StageJob J = jobs[lo];
  const LeafDesc d = leaves[J.leaf];
  const uint64_t head_bytes = d.fin_from, to = J.host ? head_bytes : d.len;
  const uint64_t m0 = (uint64_t)(blockIdx.x - J.blk_first) * kStageBytes + 16ull * threadIdx.x;
  if (m0 >= to) return;
  const char* head = reinterpret_cast<const char*>(head_table + J.head_word);
  const char* payload = reinterpret_cast<const char*>(J.payload);
  u32x4 v = {0, 0, 0, 0};
  if (m0 >= head_bytes && m0 + 16 <= to) {
    // the aligned words the sixteen bytes lie in, none of them past the payload's last
    const uint64_t src = J.payload + (m0 - head_bytes);
    const char* at = reinterpret_cast<const char*>(src & ~uint64_t(3));
    const uint32_t sh = 8 * (uint32_t)(src & 3);
    const u32x4 w = gload<u32x4w>(at);
    if (sh == 0) {
      v = w;
    } else {
      const uint32_t last = gload<uint32_t>(at + 16);
#pragma unroll
      for (int t = 0; t < 4; t++) v[t] = (w[t] >> sh) | ((t < 3 ? w[t + 1] : last) << (32 - sh));
    }
  } else {
#pragma unroll
    for (uint32_t t = 0; t < 16; t++) {
      const uint64_t m = m0 + t;
      uint32_t byte = 0;
      if (m < head_bytes) byte = gload<uint8_t>(head + m);
      else if (m < to) byte = gload<uint8_t>(payload + (m - head_bytes));
      v[t / 4] |= byte << (8 * (t % 4));
    }
  }
  gstore<u32x4>(reinterpret_cast<char*>(d.payload) + m0, v);
}

// ---- host side ----------------------------------------------------------------------------

struct HostCopy {  // a staged leaf's payload in host memory, copied into its staged message
  uint64_t dst, src, bytes;
};

struct LevelInfo {
  uint64_t ent_first;  // index of the fold's first entry in the entry array
  uint32_t n_ents;
  uint64_t n_out;
  uint64_t blk_first;  // index of the fold's block -> entry table in blk_ent
  int in_buf, out_buf;  // 0 = cv0, 1 = cv1
  bool lanes;           // level_lanes' fold, not level_kernel's
};

struct LeafPlan {
  size_t n = 0;
  uint64_t n_chunks = 0, bytes = 0;
  uint32_t n_fused = 0;  // product leaves whose P-pass sums the chunk kernel takes
  uint32_t fuse_k = 4;   // the fused plan's challenges per product (1, 2 or 4)
  uint64_t fused_msg = 0, fused_chunks = 0, fused_records = 0;  // per run of the fused kernel
  FuseDesc* d_fuse = nullptr;
  Order plain{}, fused{};  // the two kernels' chunk orders (device tables)
  bool quad = false;       // the plain order is chunk_kernel_quad's
  bool owned = false;
  char* base = nullptr;  // one device allocation: metadata, then workspace
  size_t total = 0;
  // device views
  LeafDesc* d_leaves = nullptr;
  uint32_t* d_head = nullptr;
  LevelEntry* d_levels = nullptr;
  uint32_t* d_blk_ent = nullptr;
  uint32_t* d_cv[2] = {nullptr, nullptr};
  uint32_t max_grid = 0;  // chunk kernel's grid limit; 0 = one block per slot
  std::vector<LevelInfo> levels;
  char* d_result = nullptr;  // of a synchronous call: the first-bad word (n), then the digests
  StageJob* d_stages = nullptr;
  uint32_t n_stages = 0, stage_blocks = 0;
  std::vector<HostCopy> host_copies;  // after the staging kernel
};

// Build the plan's host image and sizes. `device_only` refuses host payloads.
// A chunk order on the host: entries (first slot, leaf) and the block -> entry table.
struct OrderHost {
  std::vector<uint64_t> first;  // n_ents + 1 (closing bound = n_slots)
  std::vector<uint32_t> leaf;
  std::vector<uint32_t> blk_ent;
  uint64_t n_slots = 0;
  uint32_t n_blocks = 0;
  uint32_t run = 1, short_most = 0;  // the plain order's (lane_run)
  void add(uint32_t i, uint64_t slots) {
    first.push_back(n_slots);
    leaf.push_back(i);
    n_slots += slots;
  }
  bool finish(uint32_t per_block) {
    first.push_back(n_slots);
    const uint64_t nb = (n_slots + per_block - 1) / per_block;
    if (nb >= 0x7FFFFFFFull || leaf.size() >= 0xFFFFFFFFull) return false;
    n_blocks = (uint32_t)nb;
    blk_ent.assign(n_blocks + 1, 0);
    size_t e = 0;
    for (uint32_t b = 0; b < n_blocks; b++) {
      const uint64_t g = (uint64_t)b * per_block;
      while (first[e + 1] <= g) e++;
      blk_ent[b] = (uint32_t)e;
    }
    blk_ent[n_blocks] = leaf.empty() ? 0 : (uint32_t)(leaf.size() - 1);
    return true;
  }
};

// A fused leaf's chunk order: T classes (chunk c in class c mod T, T = lcm(row bytes, 1024) /
// 1024, so a class's chunks start at one offset in the row). A lane's run is RC = min(T, lrun)
// consecutive classes of one period, or, when T < lrun, PG = lrun / T whole periods; the runs
// of one class range get Q lanes, the number of runs rounded up to 64. Fusing is declined when
// the padding would exceed 1/16 of the chunks even with runs of one chunk.
static bool fuse_shape(uint64_t msg_bytes, uint32_t row_bytes, uint32_t lrun, uint32_t* T,
                       uint32_t* Q, uint32_t* run, uint32_t* nf, uint64_t* slots) {
  const uint64_t n_chunks = (msg_bytes + 1023) / 1024;
  const uint64_t f = msg_bytes % 1024 != 0 && msg_bytes % 1024 < 128 ? n_chunks - 1 : n_chunks;
  uint64_t a = row_bytes, b = 1024;
  while (b) {
    const uint64_t t = a % b;
    a = b;
    b = t;
  }
  const uint64_t t = (uint64_t)row_bytes / a;  // lcm / 1024
  const uint64_t periods = (f + t - 1) / t;
  // Runs of lrun chunks, or, where rounding their count up to 64 pads too much (a leaf of
  // few periods with T < lrun), runs of one chunk.
  const uint64_t shapes[2][2] = {{std::min<uint64_t>(t, lrun), t >= lrun ? 1 : lrun / t},
                                 {1, 1}};
  for (const auto& sh : shapes) {
    const uint64_t rc = sh[0], pg = sh[1];
    const uint64_t q = ((periods + pg - 1) / pg + 63) / 64 * 64;
    const uint64_t total = (t + rc - 1) / rc * q + (f < n_chunks ? 64 : 0);
    if (total >= 0xFFFFFFFFull || (t * pg * q - f) * 16 > f) continue;
    *T = (uint32_t)t;
    *Q = (uint32_t)q;
    *run = (uint32_t)(rc | pg << 16);
    *nf = (uint32_t)f;
    *slots = total;
    return true;
  }
  return false;
}

// How a plan's chunks are cut into work, by their count (one leaf of each size, MI355X, the
// chunk kernel alone; four chunks a lane / one a lane / four lanes a chunk, us):
//   6 KiB 102 / 40 / 19;  16 MiB 101 / 37 / 19;  32 MiB 110 / 35 / 26;  48 MiB 111 / 41 / 46;
//   64 MiB 109 / 42 / 54;  256 MiB 123 / 104;  384 MiB 200 / 155;  512 MiB 209 / 202;
//   1 GiB 382 / 385 / 551;  4 GiB 1444 / 1410 / 2069
// A chunk is sixteen compressions, each needing the last one's output, so below a wave for
// every SIMD (64 Ki lanes) the time is one lane's serial chain: short runs, and lanes in
// quads while those still find idle SIMDs. Runs of four save the second read of the lines
// between chunks but quarter the blocks: the GPU holds 1024 of them, each 0.4 ms long, and the
// last round of a few is part empty (a two-layer step's 6.4 M fused and 2.8 M plain chunks, 6.1
// and 2.6 rounds: 2755 and 1015 us in runs of four, 2490 and 913 singly; 8.7 M chunks in one
// plan 3010 and 2935). From kRunLeast on, sixteen rounds and more, the last one costs little.
constexpr uint64_t kQuadMost = 32768;     // chunks hashed by four lanes each, at most
constexpr uint64_t kRunLeast = 16 << 20;  // chunks from which a lane takes kRun of them
static uint32_t run_for(uint64_t chunks) { return chunks >= kRunLeast ? kRun : 1; }

// Many short leaves keep runs of kRun: a wave of single chunks goes through the header's path, the
// last block's and the whole blocks' for the sake of a few lanes each, a wave of runs once for the
// whole run. One chunk a lane / four, us, leaves at one word shift (and at all four, whose paths a
// wave of small leaves takes in turn either way), thousands of them:
//   2 chunks  64: 77 / 58 (370 / 184), 256: 261 / 175 (976 / 560);  3 chunks  43: 78 / 81
//   (267 / 278), 87: 136 / 136, 175: 267 / 219 (902 / 691);  4 chunks  64: 125 / 103 (437 / 350);
//   8 chunks  32: 137 / 136 (472 / 487), 64: 265 / 237 (884 / 814);  9 chunks  58: 262 / 319;
//   24 chunks  11: 134 / 134 (443 / 452), 44: 503 / 448 (1500 / 1451);  64 chunks  16: 470 / 418
//   (466 / 1443), 33: 933 / 810 (943 / 2782)
// So leaves of up to 24 chunks, and of up to 128 where all of them lie at one shift (with several,
// a wave of longer leaves' single chunks still has one), wherever runs take no more time by the
// rounds of 64 Ki lanes they fill (a wave on every SIMD): a run takes its blocks, a single chunk
// sixteen and an eighth more.
constexpr uint32_t kShortMixed = 24, kShortAlike = 128;

struct RunCount {
  uint64_t runs = 0, chunks = 0, blocks = 0;
  void add(uint32_t n_chunks, uint64_t bytes) {
    runs += (n_chunks + kRun - 1) / kRun;
    chunks += n_chunks;
    blocks += (bytes + 63) / 64;
  }
  bool pay() const {
    constexpr uint64_t kRound = 64 << 10;
    return runs > 0 && (double)((runs + kRound - 1) / kRound) * (double)blocks / (double)runs <=
                           (double)((chunks + kRound - 1) / kRound) * 18.0;
  }
};

static uint32_t short_for(const std::vector<LeafDesc>& desc, const std::vector<uint32_t>& leaves) {
  RunCount mixed, alike;
  uint32_t shifts = 0;
  for (uint32_t i : leaves) {
    const LeafDesc& d = desc[i];
    if (d.n_chunks < 2 || lane_run(d.n_chunks, 1, kShortAlike) != kRun) continue;
    alike.add(d.n_chunks, d.head_len + d.len);
    if (d.n_chunks <= kShortMixed) mixed.add(d.n_chunks, d.head_len + d.len);
    shifts |= 1u << ((d.payload - d.head_len) >> 2 & 3);
  }
  if ((shifts & (shifts - 1)) == 0 && alike.pay()) return kShortAlike;
  return mixed.pay() ? kShortMixed : 0;
}

// Leaves of up to kShortNodes chunks have their trees reduced a lane per eight nodes (level_lanes)
// where a plan holds kShortLeast of them or more, else a block per leaf (level_kernel), whose
// latency is shorter but which spends a block's start and the few lanes of its last levels on each.
// Lanes / blocks, us, for 2, 9, 64, 300 and 600 chunks a leaf:
//   1000 leaves 11 / 12, 22 / 12, 31 / 14, 40 / 24, 60 / 31;  4000: 12 / 13, 23 / 21, 32 / 27,
//   63 / 55, 91 / 78;  8000: 12 / 17, 23 / 32, 35 / 43, 83 / 93, 142 / 136;  16000: 12 / 26,
//   23 / 52, 46 / 76, 132 / 165;  64000: 12 / 73, 37 / 186, 106 / 267
// and for 6782 of 3 to 433 chunks among longer ones (a 135M-parameter step) 163 / 155: the line
// lies where lanes are ahead at every length up to kShortNodes.
constexpr uint64_t kShortLeast = 8000;
constexpr uint32_t kShortNodes = 512;

// Pinned memory of the synchronous entry point, per direction: a plan's metadata on the way up,
// digests on the way down. Larger ones (some 5000 leaves, 32 thousand) take pageable copies.
constexpr size_t kPinnedBytes = size_t(1) << 20;
constexpr size_t kResultHead = 16;  // bytes of a call's results before its digests

static int plan_build(size_t n, const uint8_t* hdr_buf, const uint64_t* hdr_off,
                      const uint32_t* hdr_len, const uint32_t* hdr_idx,
                      const uint64_t* payload_ptr, const uint64_t* payload_len,
                      const uint8_t* kind, bool device_only, bool owned, void* fv,
                      LeafPlan** out, char* ext_base = nullptr, size_t ext_cap = 0,
                      void* pinned = nullptr, uint32_t run_asked = 0) {
  if (n == 0 || n >= 0xFFFFFFFFull || run_asked > kRun) return POTS_E_ARG;
  for (size_t i = 0; i < n; i++)
    if (kind[i] > POTS_KIND_F16) return POTS_E_ARG;
  LeafPlan* P = new (std::nothrow) LeafPlan;
  if (!P) return POTS_E_NOMEM;
  P->n = n;
  P->owned = owned;

  // Per leaf: its head bytes (0x00 || header) and whether it must be staged.
  std::vector<LeafDesc> desc(n);
  std::vector<uint8_t> headbytes;  // word-aligned heads of direct leaves, then staged heads
  OrderHost plain, fused;
  std::vector<int64_t> stage_head_at(n, -1);
  uint64_t stage_bytes = 0, stage_blocks = 0;
  std::vector<uint64_t> stage_off(n, 0);
  std::vector<StageJob> stages;
  std::vector<FuseDesc> fdesc;                 // per fused leaf
  std::vector<uint32_t> fprod, fhead;          // its product and head bytes
  std::unordered_set<uint32_t> fused_prods;
  std::vector<uint32_t> plain_leaves;
  uint64_t plain_chunks = 0, all_chunks = 0;
  for (size_t i = 0; i < n; i++)
    all_chunks += (payload_len[i] >> 10) + 1;
  const uint32_t lrun = run_asked ? run_asked : run_for(all_chunks);
  uint64_t nc = 0;
  for (size_t i = 0; i < n; i++) {
    const uint32_t u = hdr_idx[i];
    const uint64_t hl = 1 + (uint64_t)hdr_len[u];
    const uint64_t len = payload_len[i];
    const uint64_t ptr = payload_ptr[i];
    bool host = false;
    if (len > 0) host = !is_device_pointer(reinterpret_cast<const void*>(ptr));
    if (host && device_only) {
      delete P;
      return POTS_E_ARG;
    }
    const bool stage = host || (hl % 4) != 0 || (ptr % 4) != 0;
    LeafDesc& d = desc[i];
    d.kind = kind[i];
    const uint64_t at = headbytes.size();
    headbytes.push_back(0x00);
    headbytes.insert(headbytes.end(), hdr_buf + hdr_off[u], hdr_buf + hdr_off[u] + hdr_len[u]);
    while (headbytes.size() % 4) headbytes.push_back(0);
    d.fin_from = (uint32_t)hl;  // the 0x00 || header bytes are never NaN/Inf-tested
    if (!stage) {
      d.payload = ptr;
      d.len = len;
      d.head_word = (uint32_t)(at / 4);
      d.head_len = (uint32_t)hl;
    } else {
      stage_head_at[i] = (int64_t)at;
      stage_off[i] = stage_bytes;
      stage_bytes += align_up(hl + len, 16);
      d.payload = 0;  // filled once the workspace address is known
      d.len = hl + len;
      d.head_word = 0;
      d.head_len = 0;
      const uint64_t to = host ? hl : hl + len;
      stages.push_back(StageJob{ptr, (uint32_t)i, (uint32_t)(at / 4), (uint32_t)stage_blocks,
                                host ? 1u : 0u});
      stage_blocks += (to + kStageBytes - 1) / kStageBytes;
      if (host) P->host_copies.push_back(HostCopy{stage_off[i] + hl, ptr, len});
    }
    const uint64_t L = hl + len;
    if (L >> 42) {  // 2^32 chunks: the chunk kernel's 32-bit counter
      delete P;
      return POTS_E_ARG;
    }
    const uint64_t nck = std::max<uint64_t>(1, (L + 1023) / 1024);
    d.cv_first = nc;
    d.n_chunks = (uint32_t)nck;
    d.fuse = kNoFuse;
    FusedProduct fp;
    uint32_t T = 0, Q = 0, run = 0, nf = 0;
    uint64_t slots = 0;
    if (fv && !stage && (kind[i] == POTS_KIND_BF16 || kind[i] == POTS_KIND_F32) &&
        (ptr - hl) % 16 == 4 && fv_fuse_candidate(fv, ptr, len, kind[i], &fp) &&
        !fused_prods.count(fp.prod) && fuse_shape(L, fp.w * fp.esz, lrun, &T, &Q, &run, &nf, &slots)) {
      fused_prods.insert(fp.prod);
      P->fuse_k = fp.k;  // one Freivalds plan: every fused product has the plan's k
      FuseDesc f;
      memset(&f, 0, sizeof f);
      f.r = fp.r;
      f.row_bytes = fp.w * fp.esz;
      f.n_rows = fp.n;
      f.J = (f.row_bytes + 1023) / 1024 + 1;
      f.T = T;
      f.Q = Q;
      f.esz = fp.esz;
      f.nf = nf;
      f.run = run;
      d.fuse = (uint32_t)fdesc.size();
      fdesc.push_back(f);
      fprod.push_back(fp.prod);
      fhead.push_back((uint32_t)hl);
      fused.add((uint32_t)i, slots);  // slots: a multiple of 64, so every entry is aligned
      P->fused_msg += L;
      P->fused_chunks += nck;
      {  // run records: one per (row, chunk) with elements of the row in the chunk's pairs
        const uint64_t hc = (hl + 127) & ~uint64_t(127), lf = L & ~uint64_t(127);
        for (uint64_t r = 0; r < fp.n; r++) {
          const uint64_t fs = std::max<uint64_t>(hl + r * f.row_bytes, hc);
          const uint64_t fe = std::min<uint64_t>(hl + (r + 1) * f.row_bytes, lf);
          if (fs < fe) P->fused_records += ((fe - 1) >> 10) - (fs >> 10) + 1;
        }
      }
    } else {
      plain_leaves.push_back((uint32_t)i);
      plain_chunks += nck;
    }
    nc += nck;
    P->bytes += L;
  }
  P->n_chunks = nc;
  P->n_fused = (uint32_t)fdesc.size();
  if (headbytes.size() / 4 >= 0xFFFFFFFFull || stage_blocks >= 0x7FFFFFFFull) {
    delete P;
    return POTS_E_ARG;
  }

  P->quad = !run_asked && plain_chunks <= kQuadMost;
  plain.run = P->quad ? 1 : lrun;
  if (!P->quad && !run_asked) plain.short_most = short_for(desc, plain_leaves);
  for (uint32_t i : plain_leaves) {
    const uint32_t run = lane_run(desc[i].n_chunks, plain.run, plain.short_most);
    plain.add(i, ((uint64_t)desc[i].n_chunks + run - 1) / run);
  }
  if (!plain.finish(P->quad ? kQuadChunks : kThreads) || !fused.finish(kThreads)) {
    delete P;
    return POTS_E_ARG;
  }

  // Reduction folds of kFold levels each, or kLaneFold. Level 0 nodes of leaf i sit at
  // desc[i].cv_first in cv0; a fold takes a leaf's n nodes to ceil(n / kTile) (BLAKE3's halving
  // with a promoted odd node, kFold times, composes to that ceiling), a block each, or to
  // ceil(n / kLaneTile), a lane each.
  std::vector<LevelEntry> ents;
  std::vector<uint32_t> blk_ent;
  std::vector<uint64_t> n_nodes(n), off(n);
  for (size_t i = 0; i < n; i++) {
    n_nodes[i] = desc[i].n_chunks;
    off[i] = desc[i].cv_first;
  }
  uint64_t n_short = 0;
  for (size_t i = 0; i < n; i++) n_short += n_nodes[i] >= 2 && n_nodes[i] <= kShortNodes;
  const uint32_t short_most = n_short >= kShortLeast ? kShortNodes : 0;
  std::vector<uint32_t> live[2];  // leaves of two nodes and more: level_kernel's, level_lanes'
  for (size_t i = 0; i < n; i++)
    if (n_nodes[i] >= 2) live[n_nodes[i] <= short_most].push_back((uint32_t)i);
  uint64_t cv1_need = 0;
  int in_buf = 0;
  while (!live[0].empty() || !live[1].empty()) {
    uint64_t out_next = 0;
    for (const bool lanes : {false, true}) {
      if (live[lanes].empty()) continue;
      const uint32_t fold = lanes ? kLaneFold : kFold;
      LevelInfo li{ents.size(), (uint32_t)live[lanes].size(), 0, blk_ent.size(), in_buf,
                   1 - in_buf, lanes};
      size_t left = 0;
      for (uint32_t i : live[lanes]) {
        const uint64_t nout = (n_nodes[i] + (1u << fold) - 1) >> fold;
        LevelEntry e;
        e.in_off = off[i];
        e.out_off = out_next;
        e.out_first = li.n_out;
        e.n_in = (uint32_t)n_nodes[i];
        e.leaf = i;
        ents.push_back(e);
        li.n_out += nout;
        off[i] = out_next;
        n_nodes[i] = nout;
        if (nout >= 2) {  // (a leaf that closes writes its digest and nothing else)
          out_next += nout;
          live[lanes][left++] = i;
        }
      }
      live[lanes].resize(left);
      if (li.n_out >= 0x7FFFFFFFull) {
        delete P;
        return POTS_E_ARG;
      }
      // Per block (level_kernel: one output each; level_lanes: kThreads), the fold-relative index
      // of its first output's entry; of level_lanes' a closing bound too.
      for (uint32_t k = 0; k < li.n_ents; k++) {
        const uint64_t end = k + 1 < li.n_ents ? ents[li.ent_first + k + 1].out_first : li.n_out;
        blk_ent.resize(li.blk_first + (lanes ? (end + kThreads - 1) / kThreads : end), k);
      }
      if (lanes) blk_ent.push_back(li.n_ents - 1);
      P->levels.push_back(li);
    }
    if (in_buf == 0) cv1_need = std::max(cv1_need, out_next);
    in_buf = 1 - in_buf;
  }

  // One allocation: [metadata | head table | cv0 | cv1 | staging].
  size_t at = 0;
  auto place = [&](size_t bytes) {
    size_t a = at;
    at = align_up(at + bytes, 256);
    return a;
  };
  const size_t o_leaves = place(n * sizeof(LeafDesc));
  const size_t o_fuse = place(std::max<size_t>(fdesc.size(), 1) * sizeof(FuseDesc));
  size_t o_ord[2][3];
  OrderHost* ords[2] = {&plain, &fused};
  for (int k = 0; k < 2; k++) {
    o_ord[k][0] = place(ords[k]->first.size() * sizeof(uint64_t));
    o_ord[k][1] = place(std::max<size_t>(ords[k]->leaf.size(), 1) * sizeof(uint32_t));
    o_ord[k][2] = place(ords[k]->blk_ent.size() * sizeof(uint32_t));
  }
  const size_t o_head = place(std::max<size_t>(headbytes.size(), 4));
  const size_t o_lev = place(std::max<size_t>(ents.size(), 1) * sizeof(LevelEntry));
  const size_t o_blk_ent = place(std::max<size_t>(blk_ent.size(), 1) * sizeof(uint32_t));
  // The staging jobs last: a call that runs once, in memory it must fit, has them where its chunk
  // kernels then put the chaining values, which take more (32 bytes a chunk).
  const size_t o_stages = at, stages_bytes = stages.size() * sizeof(StageJob);
  if (!ext_base) place(stages_bytes);
  // A synchronous call's results: the first-bad word, uploaded with the metadata as n, and the
  // digests behind it, so that one copy brings both back.
  size_t o_bad = 0, meta_bytes = o_stages + stages_bytes;
  if (pinned) {
    o_bad = place(kResultHead + 32 * n);
    meta_bytes = o_bad + kResultHead;
  }
  const size_t o_cv0 = place(nc * 32);
  const size_t o_cv1 = place(std::max<uint64_t>(cv1_need, 1) * 32);
  const size_t o_stage = place(std::max<uint64_t>(stage_bytes, 16));
  P->total = at;

  int rc;
  if (ext_base) {  // memory the caller holds (the allocation-free entry point's scratch)
    if (P->total > ext_cap) {
      note_error("leaf hashing needs " + std::to_string(P->total) + " bytes of device scratch "
                 "for these leaves; the allocation-free entry point holds " +
                 std::to_string(ext_cap));
      delete P;
      return POTS_E_ARG;
    }
    P->owned = false;
    P->base = ext_base;
  } else if (owned) {
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&P->base), P->total);
    if (e != hipSuccess) {
      note_hip_error(e, "hipMalloc(leaf plan)", __FILE__, __LINE__);
      delete P;
      return e == hipErrorOutOfMemory ? POTS_E_NOMEM : POTS_E_HIP;
    }
  } else {
    void* p = nullptr;
    if ((rc = arena_get(0, P->total, &p)) != POTS_E_OK) {
      delete P;
      return rc;
    }
    P->base = static_cast<char*>(p);
  }
  const uint64_t B = reinterpret_cast<uint64_t>(P->base);
  for (size_t i = 0; i < n; i++)
    if (stage_head_at[i] >= 0) desc[i].payload = B + o_stage + stage_off[i];
  for (HostCopy& c : P->host_copies) c.dst += B + o_stage;
  P->d_stages = reinterpret_cast<StageJob*>(P->base + o_stages);
  P->n_stages = (uint32_t)stages.size();
  P->stage_blocks = (uint32_t)stage_blocks;
  P->d_leaves = reinterpret_cast<LeafDesc*>(P->base + o_leaves);
  P->d_fuse = reinterpret_cast<FuseDesc*>(P->base + o_fuse);
  Order* dords[2] = {&P->plain, &P->fused};
  for (int k = 0; k < 2; k++) {
    dords[k]->first = reinterpret_cast<const uint64_t*>(P->base + o_ord[k][0]);
    dords[k]->leaf = reinterpret_cast<const uint32_t*>(P->base + o_ord[k][1]);
    dords[k]->blk_ent = reinterpret_cast<const uint32_t*>(P->base + o_ord[k][2]);
    dords[k]->n_slots = ords[k]->n_slots;
    dords[k]->n_blocks = ords[k]->n_blocks;
    dords[k]->run = ords[k]->run;
    dords[k]->short_most = ords[k]->short_most;
  }
  P->d_head = reinterpret_cast<uint32_t*>(P->base + o_head);
  P->d_levels = reinterpret_cast<LevelEntry*>(P->base + o_lev);
  P->d_blk_ent = reinterpret_cast<uint32_t*>(P->base + o_blk_ent);
  P->d_cv[0] = reinterpret_cast<uint32_t*>(P->base + o_cv0);
  P->d_cv[1] = reinterpret_cast<uint32_t*>(P->base + o_cv1);

  // The fused products' run records, allocated by the Freivalds plan.
  if (!fdesc.empty()) {
    std::vector<uint64_t> segs;
    const int frc = fv_fuse_commit(fv, fprod, fhead, &segs);
    if (frc != POTS_E_OK) {
      if (owned) (void)hipFree(P->base);
      delete P;
      return frc;
    }
    for (size_t f = 0; f < fdesc.size(); f++) fdesc[f].seg = segs[f];
  }

  // Upload the metadata in one copy; from pinned memory of kPinnedBytes, if given, in the null
  // stream's order, the caller waiting for that stream before it lets the memory go.
  std::vector<char> img(meta_bytes, 0);
  memcpy(img.data() + o_leaves, desc.data(), n * sizeof(LeafDesc));
  if (!fdesc.empty()) memcpy(img.data() + o_fuse, fdesc.data(), fdesc.size() * sizeof(FuseDesc));
  for (int k = 0; k < 2; k++) {
    memcpy(img.data() + o_ord[k][0], ords[k]->first.data(),
           ords[k]->first.size() * sizeof(uint64_t));
    if (!ords[k]->leaf.empty())
      memcpy(img.data() + o_ord[k][1], ords[k]->leaf.data(),
             ords[k]->leaf.size() * sizeof(uint32_t));
    memcpy(img.data() + o_ord[k][2], ords[k]->blk_ent.data(),
           ords[k]->blk_ent.size() * sizeof(uint32_t));
  }
  if (!stages.empty()) memcpy(img.data() + o_stages, stages.data(), stages_bytes);
  if (!headbytes.empty()) memcpy(img.data() + o_head, headbytes.data(), headbytes.size());
  if (!ents.empty()) memcpy(img.data() + o_lev, ents.data(), ents.size() * sizeof(LevelEntry));
  if (!blk_ent.empty())
    memcpy(img.data() + o_blk_ent, blk_ent.data(), blk_ent.size() * sizeof(uint32_t));
  if (pinned) {
    const uint32_t none = (uint32_t)n;
    memcpy(img.data() + o_bad, &none, 4);
    P->d_result = P->base + o_bad;
  }
  hipError_t e;
  if (pinned && meta_bytes <= kPinnedBytes) {
    memcpy(pinned, img.data(), meta_bytes);
    e = hipMemcpyAsync(P->base, pinned, meta_bytes, hipMemcpyHostToDevice, 0);
  } else {
    e = hipMemcpy(P->base, img.data(), meta_bytes, hipMemcpyHostToDevice);
  }
  if (e != hipSuccess) {
    note_hip_error(e, "hipMemcpy(leaf plan metadata)", __FILE__, __LINE__);
    if (owned) (void)hipFree(P->base);
    delete P;
    return POTS_E_HIP;
  }
  *out = P;
  return POTS_E_OK;
}

// One stage of a plan's run: 0 staging copies and the first-bad reset, 1 the chunk kernel,
// 2 the per-leaf tree levels.
static int plan_stage(LeafPlan* P, int stage, uint32_t* d_digests, uint32_t* d_first_bad,
                      hipStream_t stream) {
  int rc;
  switch (stage) {
    case 0:
      hipLaunchKernelGGL(stage_kernel, dim3(std::max(1u, P->stage_blocks)), dim3(kThreads), 0,
                         stream, P->d_stages, P->n_stages, P->d_leaves, P->d_head, d_first_bad,
                         (uint32_t)P->n);
      for (const HostCopy& c : P->host_copies)
        POTS_HIP(hipMemcpyAsync(reinterpret_cast<void*>(c.dst), reinterpret_cast<const void*>(c.src),
                                c.bytes, hipMemcpyHostToDevice, stream));
      POTS_HIP(hipGetLastError());
      return POTS_E_OK;
    case 1:  // both chunk kernels: the fused leaves' (3), then the others' (4)
      if ((rc = plan_stage(P, POTS_LEAF_STAGE_FUSED_CHUNKS, d_digests, d_first_bad, stream)) !=
          POTS_E_OK)
        return rc;
      return plan_stage(P, POTS_LEAF_STAGE_PLAIN_CHUNKS, d_digests, d_first_bad, stream);
    case POTS_LEAF_STAGE_FUSED_CHUNKS:
      if (P->fused.n_blocks) {
        const dim3 grid(P->max_grid ? std::min(P->max_grid, P->fused.n_blocks)
                                    : P->fused.n_blocks);
        switch (P->fuse_k) {
          case 1:
            hipLaunchKernelGGL(chunk_kernel_fused<1>, grid, dim3(kThreads), 0, stream,
                               P->d_leaves, P->d_fuse, P->fused, P->d_head, P->d_cv[0],
                               d_first_bad);
            break;
          case 2:
            hipLaunchKernelGGL(chunk_kernel_fused<2>, grid, dim3(kThreads), 0, stream,
                               P->d_leaves, P->d_fuse, P->fused, P->d_head, P->d_cv[0],
                               d_first_bad);
            break;
          case 4:
            hipLaunchKernelGGL(chunk_kernel_fused<4>, grid, dim3(kThreads), 0, stream,
                               P->d_leaves, P->d_fuse, P->fused, P->d_head, P->d_cv[0],
                               d_first_bad);
            break;
          default:
            return POTS_E_ARG;
        }
        POTS_HIP(hipGetLastError());
      }
      return POTS_E_OK;
    case POTS_LEAF_STAGE_PLAIN_CHUNKS:
      if (P->plain.n_blocks && P->quad) {
        // a limit counts blocks of 256 lanes, four of this kernel's
        const uint64_t most = P->max_grid ? 4ull * P->max_grid : P->plain.n_blocks;
        hipLaunchKernelGGL(chunk_kernel_quad,
                           dim3((uint32_t)std::min<uint64_t>(most, P->plain.n_blocks)), dim3(64),
                           0, stream, P->d_leaves, P->plain, P->d_head, P->d_cv[0], d_digests,
                           d_first_bad);
        POTS_HIP(hipGetLastError());
      } else if (P->plain.n_blocks) {
        hipLaunchKernelGGL(chunk_kernel,
                           dim3(P->max_grid ? std::min(P->max_grid, P->plain.n_blocks)
                                            : P->plain.n_blocks),
                           dim3(kThreads), 0, stream, P->d_leaves, P->plain, P->d_head,
                           P->d_cv[0], d_digests, d_first_bad);
        POTS_HIP(hipGetLastError());
      }
      return POTS_E_OK;
    case 2:
      for (const LevelInfo& li : P->levels) {
        if (li.lanes)
          hipLaunchKernelGGL(level_lanes, dim3((uint32_t)((li.n_out + kThreads - 1) / kThreads)),
                             dim3(kThreads), 0, stream, P->d_levels + li.ent_first,
                             P->d_blk_ent + li.blk_first, li.n_out, P->d_cv[li.in_buf],
                             P->d_cv[li.out_buf], d_digests);
        else
          hipLaunchKernelGGL(level_kernel, dim3((uint32_t)li.n_out), dim3(kThreads), 0, stream,
                             P->d_levels + li.ent_first, P->d_blk_ent + li.blk_first,
                             P->d_cv[li.in_buf], P->d_cv[li.out_buf], d_digests);
        POTS_HIP(hipGetLastError());
      }
      return POTS_E_OK;
    default:
      return POTS_E_ARG;
  }
}

static int plan_run(LeafPlan* P, uint32_t* d_digests, uint32_t* d_first_bad,
                    hipStream_t stream) {
  for (int stage = 0; stage < POTS_LEAF_STAGES; stage++) {
    const int rc = plan_stage(P, stage, d_digests, d_first_bad, stream);
    if (rc != POTS_E_OK) return rc;
  }
  return POTS_E_OK;
}

static void plan_free(LeafPlan* P) {
  if (!P) return;
  if (P->owned && P->base) (void)hipFree(P->base);
  delete P;
}

}  // namespace pots

using namespace pots;

extern "C" size_t pots_hash_leaves(size_t n, const uint8_t* hdr_buf, const uint64_t* hdr_off,
                                   const uint32_t* hdr_len, const uint32_t* hdr_idx,
                                   const uint64_t* payload_ptr, const uint64_t* payload_len,
                                   const uint8_t* kind, uint8_t* out, uint32_t n_threads) {
  (void)n_threads;
  if (n == 0) return 0;
  // One call at a time: they share the arenas and the pinned memory. A small call's metadata and
  // digests go through pinned memory, one copy each way in the null stream's order and one wait
  // at the end (three pageable copies, each waited for, were 30 us of a norm's leaf hash).
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  void* pinned = nullptr;
  if (pinned_get(0, 2 * kPinnedBytes, &pinned) != POTS_E_OK) {
    pinned = nullptr;
    (void)hipGetLastError();  // pageable copies instead: the next launch's check is not to see it
  }
  LeafPlan* P = nullptr;
  void* res = nullptr;
  size_t bad = SIZE_MAX;
  const size_t res_bytes = kResultHead + 32 * n;
  if (plan_build(n, hdr_buf, hdr_off, hdr_len, hdr_idx, payload_ptr, payload_len, kind,
                 /*device_only=*/false, /*owned=*/false, nullptr, &P, nullptr, 0, pinned) ==
          POTS_E_OK &&
      (P->d_result || arena_get(1, res_bytes, &res) == POTS_E_OK)) {
    char* d_res = P->d_result ? P->d_result : static_cast<char*>(res);
    uint32_t* d_bad = reinterpret_cast<uint32_t*>(d_res);
    uint32_t* d_dig = reinterpret_cast<uint32_t*>(d_res + kResultHead);
    // the staging stage only where there is something to stage or a first-bad word to reset
    int rc = POTS_E_OK;
    for (int stage = P->d_result && P->n_stages == 0 ? 1 : 0;
         stage < POTS_LEAF_STAGES && rc == POTS_E_OK; stage++)
      rc = plan_stage(P, stage, d_dig, d_bad, 0);
    if (rc == POTS_E_OK) {
      uint32_t h_bad = 0;
      hipError_t e;
      if (pinned && res_bytes <= kPinnedBytes) {
        char* back = static_cast<char*>(pinned) + kPinnedBytes;
        e = hipMemcpyAsync(back, d_res, res_bytes, hipMemcpyDeviceToHost, 0);
        if (e == hipSuccess) e = hipStreamSynchronize(0);
        if (e == hipSuccess) {
          memcpy(&h_bad, back, 4);
          memcpy(out, back + kResultHead, 32 * n);
        }
      } else {
        e = hipMemcpy(out, d_dig, 32 * n, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(&h_bad, d_bad, 4, hipMemcpyDeviceToHost);
      }
      if (e == hipSuccess) bad = h_bad;
      else note_hip_error(e, "hipMemcpy(digests)", __FILE__, __LINE__);
    }
  }
  if (bad == SIZE_MAX) (void)hipStreamSynchronize(0);  // a copy from the pinned memory may be left
  plan_free(P);
  return bad;
}

// ---- the allocation-free variant of pots_hash_leaves ----------------------------------------

// Device scratch of pots_hash_leaves_noalloc: the results (32 B per leaf and the first-bad
// word), then the plan (leaf descriptors, chaining values, staged messages). Each GPU the
// library runs on holds its own copy until the process ends.
constexpr size_t kNoallocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kNoallocScratchBytes];

namespace {
std::mutex g_scratch_mu;  // one call at a time per process: every call shares the array
char* g_scratch_ptr[64] = {};

// The array's device address on the current GPU, looked up once per device with that device
// current. Host code passes this address, never the symbol itself.
int scratch_address(char** out) {
  int dev = 0;
  POTS_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return POTS_E_ARG;
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      note_hip_error(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
      return POTS_E_HIP;
    }
    g_scratch_ptr[dev] = static_cast<char*>(p);
  }
  *out = g_scratch_ptr[dev];
  return POTS_E_OK;
}
}  // namespace

extern "C" size_t pots_hash_leaves_noalloc(size_t n, const uint8_t* hdr_buf,
                                           const uint64_t* hdr_off, const uint32_t* hdr_len,
                                           const uint32_t* hdr_idx, const uint64_t* payload_ptr,
                                           const uint64_t* payload_len, const uint8_t* kind,
                                           uint8_t* out, uint32_t n_threads) {
  (void)n_threads;
  if (n == 0) return 0;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  char* base = nullptr;
  if (scratch_address(&base) != POTS_E_OK) return SIZE_MAX;
  const size_t res_bytes = align_up(32 * n + 16, 256);
  if (res_bytes >= kNoallocScratchBytes) {
    note_error(std::to_string(n) + " leaves need " + std::to_string(res_bytes) + " bytes of "
               "results; the allocation-free entry point's scratch holds " +
               std::to_string(kNoallocScratchBytes));
    return SIZE_MAX;
  }
  // In runs of kRun, whose tables are the smallest, where the plan's own cut does not fit.
  LeafPlan* P = nullptr;
  int rc = POTS_E_ARG;
  for (uint32_t run = 0; run <= kRun && rc == POTS_E_ARG; run += kRun)
    rc = plan_build(n, hdr_buf, hdr_off, hdr_len, hdr_idx, payload_ptr, payload_len, kind,
                    /*device_only=*/false, /*owned=*/false, nullptr, &P, base + res_bytes,
                    kNoallocScratchBytes - res_bytes, nullptr, run);
  if (rc != POTS_E_OK) return SIZE_MAX;
  uint32_t* d_dig = reinterpret_cast<uint32_t*>(base);
  uint32_t* d_bad = reinterpret_cast<uint32_t*>(base + 32 * n);
  size_t bad = SIZE_MAX;
  uint32_t h_bad = 0;
  if (plan_run(P, d_dig, d_bad, 0) == POTS_E_OK) {
    hipError_t e = hipMemcpy(out, d_dig, 32 * n, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(&h_bad, d_bad, 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) bad = h_bad;
    else note_hip_error(e, "hipMemcpy(digests)", __FILE__, __LINE__);
  }
  plan_free(P);  // host bookkeeping only: the plan's memory is the scratch
  return bad;
}

extern "C" int pots_leaf_plan_create(size_t n, const uint8_t* hdr_buf, const uint64_t* hdr_off,
                                     const uint32_t* hdr_len, const uint32_t* hdr_idx,
                                     const uint64_t* payload_ptr, const uint64_t* payload_len,
                                     const uint8_t* kind, void** plan) {
  if (!plan) return POTS_E_ARG;
  LeafPlan* P = nullptr;
  int rc = plan_build(n, hdr_buf, hdr_off, hdr_len, hdr_idx, payload_ptr, payload_len, kind,
                      /*device_only=*/true, /*owned=*/true, nullptr, &P);
  if (rc == POTS_E_OK) *plan = P;
  return rc;
}

extern "C" int pots_leaf_plan_create_fused(size_t n, const uint8_t* hdr_buf,
                                           const uint64_t* hdr_off, const uint32_t* hdr_len,
                                           const uint32_t* hdr_idx, const uint64_t* payload_ptr,
                                           const uint64_t* payload_len, const uint8_t* kind,
                                           void* fv_plan, void** plan) {
  if (!plan || !fv_plan) return POTS_E_ARG;
  LeafPlan* P = nullptr;
  int rc = plan_build(n, hdr_buf, hdr_off, hdr_len, hdr_idx, payload_ptr, payload_len, kind,
                      /*device_only=*/true, /*owned=*/true, fv_plan, &P);
  if (rc == POTS_E_OK) *plan = P;
  return rc;
}

extern "C" int pots_leaf_plan_create_runs(size_t n, const uint8_t* hdr_buf,
                                          const uint64_t* hdr_off, const uint32_t* hdr_len,
                                          const uint32_t* hdr_idx, const uint64_t* payload_ptr,
                                          const uint64_t* payload_len, const uint8_t* kind,
                                          void* fv_plan, uint32_t run, void** plan) {
  if (!plan) return POTS_E_ARG;
  LeafPlan* P = nullptr;
  int rc = plan_build(n, hdr_buf, hdr_off, hdr_len, hdr_idx, payload_ptr, payload_len, kind,
                      /*device_only=*/true, /*owned=*/true, fv_plan, &P, nullptr, 0, nullptr, run);
  if (rc == POTS_E_OK) *plan = P;
  return rc;
}

extern "C" uint32_t pots_leaf_plan_fused(const void* plan) {
  return plan ? static_cast<const LeafPlan*>(plan)->n_fused : 0;
}

extern "C" int pots_leaf_plan_fused_stats(const void* plan, uint64_t* msg_bytes,
                                          uint64_t* chunks, uint64_t* records) {
  if (!plan || !msg_bytes || !chunks || !records) return POTS_E_ARG;
  const LeafPlan* P = static_cast<const LeafPlan*>(plan);
  *msg_bytes = P->fused_msg;
  *chunks = P->fused_chunks;
  *records = P->fused_records;
  return POTS_E_OK;
}

extern "C" int pots_step_run(void* leaf_plan, void* fv_plan, const uint8_t* d_key,
                             uint8_t* d_digests, uint32_t* d_first_bad, double* d_rows,
                             void* stream) {
  if (!leaf_plan || !fv_plan || !d_key || !d_digests || !d_first_bad || !d_rows)
    return POTS_E_ARG;
  int rc;
  if ((rc = pots_fv_plan_run_stage(fv_plan, 0, d_key, d_rows, stream)) != POTS_E_OK) return rc;
  for (int st = 0; st < POTS_LEAF_STAGES; st++)
    if ((rc = pots_leaf_plan_run_stage(leaf_plan, st, d_digests, d_first_bad, stream)) !=
        POTS_E_OK)
      return rc;
  for (int st = 1; st < POTS_FV_STAGES; st++)
    if ((rc = pots_fv_plan_run_stage(fv_plan, st, d_key, d_rows, stream)) != POTS_E_OK)
      return rc;
  return POTS_E_OK;
}

extern "C" int pots_leaf_plan_run(void* plan, uint8_t* d_out, uint32_t* d_first_bad,
                                  void* stream) {
  if (!plan || !d_out || !d_first_bad) return POTS_E_ARG;
  return plan_run(static_cast<LeafPlan*>(plan), reinterpret_cast<uint32_t*>(d_out),
                  d_first_bad, static_cast<hipStream_t>(stream));
}

extern "C" int pots_leaf_plan_run_stage(void* plan, int stage, uint8_t* d_out,
                                        uint32_t* d_first_bad, void* stream) {
  if (!plan || !d_out || !d_first_bad || stage < 0 ||
      stage > POTS_LEAF_STAGE_PLAIN_CHUNKS)
    return POTS_E_ARG;
  return plan_stage(static_cast<LeafPlan*>(plan), stage, reinterpret_cast<uint32_t*>(d_out),
                    d_first_bad, static_cast<hipStream_t>(stream));
}

extern "C" int pots_leaf_plan_set_grid(void* plan, uint32_t max_blocks) {
  if (!plan) return POTS_E_ARG;
  static_cast<LeafPlan*>(plan)->max_grid = max_blocks;
  return POTS_E_OK;
}

extern "C" uint64_t pots_leaf_plan_chunks(const void* plan) {
  return plan ? static_cast<const LeafPlan*>(plan)->n_chunks : 0;
}

extern "C" uint64_t pots_leaf_plan_bytes(const void* plan) {
  return plan ? static_cast<const LeafPlan*>(plan)->bytes : 0;
}

extern "C" void pots_leaf_plan_destroy(void* plan) { plan_free(static_cast<LeafPlan*>(plan)); }
