// Check 6a on gfx950: the SGD update identity of every linear weight, from its committed
// leaves, in one streaming pass.
//
// Reference: verification/verifier/checks.py:380-451 (_update_identity,
// _update_identity_reference) and :301-377 (_fast_rho_max), with the weight's gradient
// G = chain_gradient(its weight-gradient product leaves) (verification/computation/
// interface.py:169-180): the parts widened to fp32 and added in order. Per entry i, in fp32
// with every operation rounded on its own (no contraction), as the reference's torch ops
// round them:
//   ηG_i = fl(η·G_i),  R_i = |W_{t+1,i} − (W_t,i − ηG_i)|,  scale_i = fl(ε_W·(|W_t,i| + |ηG_i|))
// and ρ_i = 0 when R_i = 0, else fl64(R_i) / fl64(scale_i). Per weight the kernel returns
// ρ_max (the maximum, NaN if any ρ_i is NaN, as torch's max), the first index whose R_i or
// scale_i is not finite, and the first index whose ρ_i is not ≤ τ_W; the host words the
// reference's rejection from those.
//
// Bound by HBM. Work split: a block of 256 threads takes 16384 consecutive entries of one
// weight in four steps; a thread takes four groups of four entries per step, neighbouring
// threads neighbouring groups, so every load of a wave is one contiguous span, and all of a
// step's loads go out before its arithmetic (4-byte loads where a pointer is not 16-byte
// aligned, and for a weight's last partial step). A block reduces its maximum and first indices
// and makes at most one atomic update per output. Four layers' weights with bf16 gradients
// (1.87 GB): 604 us when a thread took 8 consecutive entries and every wave of 2048 entries
// updated the weight's maximum, 317 us (5.9 TB/s, what a plain read reaches) now; atomics per
// block and 8192, 16384 or 32768 entries a block: 339, 317, 319. ρ_max is kept as the bit
// pattern of a non-negative double, whose unsigned order is its numeric order with NaN above
// +inf.
#include <math.h>
#include <string.h>

#include <new>
#include <vector>

#include "common.h"
#include "gmem.h"

namespace pots {

constexpr uint32_t kUpdThreads = 256;
constexpr uint32_t kUpdGroups = 4;  // four-entry groups a thread takes per step
constexpr uint32_t kUpdSteps = 4;   // steps per block
// Groups and steps by a plan's entries, for enough blocks: 1024 entries a block (one group, one
// step) below kUpdSmall, 4096 (one step) below kUpdWide, else 16384. Both kernels of a run, us,
// before (8192 a block, an atomic per wave) and now: 0.56 M entries 11.0 -> 10.0, 1.9 M
// 13.3 -> 9.7 (17.3 at 1024 a block), 6.0 M 26 -> 20, 15 M 76 -> 33, 61 M 178 -> 117.
constexpr uint64_t kUpdSmall = 1 << 20, kUpdWide = 8 << 20;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float v4f32 __attribute__((ext_vector_type(4)));

struct UpdJob {
  uint64_t w_t, w_next;                    // fp32 [n]
  uint64_t parts[POTS_UPDATE_MAX_PARTS];   // gradient parts, [n] each
  uint32_t part_dt[POTS_UPDATE_MAX_PARTS]; // 0 fp32, 1 bf16
  uint32_t n_parts, vec;  // vec: every pointer 16-byte aligned (vector loads)
  uint64_t n;
  uint64_t block_first;
  double tau_w;
};

struct UpdOut {  // per weight, device side
  uint64_t rho_bits;
  uint64_t first_nonfinite;
  uint64_t first_over;
};
static_assert(sizeof(UpdOut) == sizeof(pots_update_result), "result layout");

__device__ __forceinline__ float load_part(uint64_t base, uint32_t dt, uint64_t i) {
  if (dt == 1) return __uint_as_float((uint32_t)gload<uint16_t>(reinterpret_cast<const uint16_t*>(base) + i) << 16);
  return gload<float>(reinterpret_cast<const float*>(base) + i);
}

__global__ __launch_bounds__(kUpdThreads) void update_init(UpdOut* __restrict__ out, uint32_t n) {
  const uint32_t t = blockIdx.x * kUpdThreads + threadIdx.x;
  if (t < n) {
    out[t].rho_bits = 0;
    out[t].first_nonfinite = ~0ull;
    out[t].first_over = ~0ull;
  }
}

// The per-thread state of the reduction, without a division per entry. The entry with the
// largest r/s is kept as its r and s and compared by cross products, exact in fp64 (24 bits
// times 24 bits); rounding is monotone, so the one quotient taken at the end is the maximum of
// the quotients. An entry lies within tau_w if r <= tau_lo·s, tau_lo a hair under tau_w; one
// that does not pass that test, or is not finite, has its quotient taken.
struct UpdAcc {
  float r = 0.f, s = 1.f;  // the largest ratio of finite entries
  double rho_max = 0.0;    // of the entries that were divided
  bool nan_seen = false;
  uint64_t first_nf = ~0ull, first_over = ~0ull;
  __device__ __forceinline__ void add(float w, float w1, float g, float eta, float eps_w,
                                      double tau_w, double tau_lo, uint64_t i) {
    const float eg = eta * g;
    const float ri = fabsf(w1 - (w - eg));
    const float si = eps_w * (fabsf(w) + fabsf(eg));
    const double rd = (double)ri, sd = (double)si;
    // false for a NaN r, a NaN s and a NaN or negative tau_lo; false for an infinite r too, since
    // tau_lo is bounded so that no finite s takes tau_lo·s to infinity; an infinite s passes with
    // any r but a NaN, so it is tested on its own
    if (rd <= tau_lo * sd && si < INFINITY) {
      if (rd * (double)s > (double)r * sd) {
        r = ri;
        s = si;
      }
      return;
    }
    if (!(isfinite(ri) && isfinite(si)) && i < first_nf) first_nf = i;
    const double rho = ri == 0.f ? 0.0 : rd / sd;
    if (rho != rho) nan_seen = true;
    else if (rho > rho_max) rho_max = rho;
    if (!(rho <= tau_w) && i < first_over) first_over = i;
  }
  __device__ __forceinline__ uint64_t rho_bits() const {
    if (nan_seen) return 0x7FF8000000000000ull;
    const double rho = r == 0.f ? 0.0 : (double)r / (double)s;
    return (uint64_t)__double_as_longlong(rho > rho_max ? rho : rho_max);
  }
};

// Four consecutive entries of a gradient part.
__device__ __forceinline__ v4f32 load4_part(uint64_t base, uint32_t dt, uint64_t i) {
  if (dt != 1) return gload<v4f32>(reinterpret_cast<const float*>(base) + i);
  const u32x2 a = gload<u32x2>(reinterpret_cast<const uint16_t*>(base) + i);
  return v4f32{__uint_as_float(a.x << 16), __uint_as_float(a.x & 0xFFFF0000u),
               __uint_as_float(a.y << 16), __uint_as_float(a.y & 0xFFFF0000u)};
}

template <uint32_t G, uint32_t STEPS>
__global__ __launch_bounds__(kUpdThreads) void update_kernel(const UpdJob* __restrict__ jobs,
                                                             const uint32_t* __restrict__ blk_job,
                                                             float eta, float eps_w,
                                                             UpdOut* __restrict__ out) {
  const uint32_t ji = blk_job[blockIdx.x];
  const UpdJob& J = jobs[ji];
  const uint64_t n = J.n;
  constexpr uint32_t kStep = kUpdThreads * 4 * G;  // entries per step
  const uint64_t base = (uint64_t)(blockIdx.x - J.block_first) * kStep * STEPS;
  const float* wt = reinterpret_cast<const float*>(J.w_t);
  const float* wn = reinterpret_cast<const float*>(J.w_next);
  // (relative error of tau_lo·s under 2^-51: r <= tau_lo·s means r/s < tau_w exactly, and a
  // product too small to be normal is below every nonzero r. A band past 2^800 tests as 2^800: no
  // ratio of finite fp32 values but r/0 comes near it, and 2^800 times an fp32 s is finite, so an
  // infinite r is never within it, whatever the band.)
  const double tau_w = J.tau_w;
  const double tau_lo = tau_w >= 0 ? fmin(tau_w, 0x1p800) * (1.0 - 0x1p-50) : __builtin_nan("");
  UpdAcc acc;
#pragma unroll 1
  for (uint32_t st = 0; st < STEPS; st++) {
    const uint64_t b0 = base + (uint64_t)st * kStep;
    if (b0 >= n) break;
    if (J.vec && b0 + kStep <= n) {
      v4f32 w[G], w1[G], g[G];
#pragma unroll
      for (uint32_t h = 0; h < G; h++) {
        const uint64_t i = b0 + 4 * (threadIdx.x + kUpdThreads * h);
        w[h] = gload<v4f32>(wt + i);
        w1[h] = gload<v4f32>(wn + i);
        g[h] = load4_part(J.parts[0], J.part_dt[0], i);
      }
      for (uint32_t p = 1; p < J.n_parts; p++)
#pragma unroll
        for (uint32_t h = 0; h < G; h++) {
          const v4f32 x = load4_part(J.parts[p], J.part_dt[p],
                                     b0 + 4 * (threadIdx.x + kUpdThreads * h));
#pragma unroll
          for (int e = 0; e < 4; e++) g[h][e] = g[h][e] + x[e];
        }
#pragma unroll
      for (uint32_t h = 0; h < G; h++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          acc.add(w[h][e], w1[h][e], g[h][e], eta, eps_w, tau_w, tau_lo,
                  b0 + 4 * (threadIdx.x + kUpdThreads * h) + e);
    } else {
      for (uint32_t h = 0; h < G; h++) {
        const uint64_t i = b0 + 4 * (threadIdx.x + kUpdThreads * h);
        if (J.vec && i + 4 <= n) {
          const v4f32 w = gload<v4f32>(wt + i), w1 = gload<v4f32>(wn + i);
          v4f32 g = load4_part(J.parts[0], J.part_dt[0], i);
          for (uint32_t p = 1; p < J.n_parts; p++) {
            const v4f32 x = load4_part(J.parts[p], J.part_dt[p], i);
#pragma unroll
            for (int e = 0; e < 4; e++) g[e] = g[e] + x[e];
          }
#pragma unroll
          for (int e = 0; e < 4; e++)
            acc.add(w[e], w1[e], g[e], eta, eps_w, tau_w, tau_lo, i + e);
          continue;
        }
        for (uint64_t t = i; t < i + 4 && t < n; t++) {
          float g = load_part(J.parts[0], J.part_dt[0], t);
          for (uint32_t p = 1; p < J.n_parts; p++) g = g + load_part(J.parts[p], J.part_dt[p], t);
          acc.add(gload<float>(wt + t), gload<float>(wn + t), g, eta, eps_w, tau_w, tau_lo, t);
        }
      }
    }
  }
  uint64_t bits = acc.rho_bits();
  uint64_t first_nf = acc.first_nf, first_over = acc.first_over;
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t b2 = __shfl_xor(bits, o);
    const uint64_t f2 = __shfl_xor(first_nf, o);
    const uint64_t v2 = __shfl_xor(first_over, o);
    bits = b2 > bits ? b2 : bits;
    first_nf = f2 < first_nf ? f2 : first_nf;
    first_over = v2 < first_over ? v2 : first_over;
  }
  // The block's thread 0 updates the weight's outputs, and only where they change: a weight's
  // blocks share one address, and atomics from every wave of them (one per 2048 entries) took
  // longer than the reads.
  __shared__ uint64_t s_out[kUpdThreads / 64][3];
  if ((threadIdx.x & 63) == 0) {
    uint64_t* w = s_out[threadIdx.x >> 6];
    w[0] = bits;
    w[1] = first_nf;
    w[2] = first_over;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (uint32_t w = 1; w < kUpdThreads / 64; w++) {
    bits = s_out[w][0] > bits ? s_out[w][0] : bits;
    first_nf = s_out[w][1] < first_nf ? s_out[w][1] : first_nf;
    first_over = s_out[w][2] < first_over ? s_out[w][2] : first_over;
  }
  unsigned long long* o = reinterpret_cast<unsigned long long*>(out + ji);
  if (bits > __hip_atomic_load(o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(o, (unsigned long long)bits);
  if (first_nf != ~0ull) atomicMin(o + 1, (unsigned long long)first_nf);
  if (first_over != ~0ull) atomicMin(o + 2, (unsigned long long)first_over);
}

struct UpdatePlan {
  size_t n = 0;
  float eta = 0.f, eps_w = 0.f;
  char* base = nullptr;
  UpdJob* d_jobs = nullptr;
  uint32_t* d_blk = nullptr;
  uint32_t n_blocks = 0;
  uint32_t groups = 1, steps = 1;  // of update_kernel
  uint64_t bytes = 0;  // algorithmic bytes read per run
};

}  // namespace pots

using namespace pots;

extern "C" int pots_update_plan_create(size_t n, const pots_update_weight* weights, float eta,
                                       float eps_w, void** plan) {
  if (!plan || !weights || n == 0 || n >= 0x7FFFFFFFull) return POTS_E_ARG;
  if (!(eta > 0.f) || !isfinite(eta) || !(eps_w > 0.f) || !isfinite(eps_w)) return POTS_E_ARG;
  std::vector<UpdJob> jobs(n);
  std::vector<uint32_t> blk;
  uint64_t bytes = 0, entries = 0;
  for (size_t i = 0; i < n; i++) entries += weights[i].n;
  const uint32_t groups = entries < kUpdSmall ? 1 : kUpdGroups;
  const uint32_t steps = entries < kUpdWide ? 1 : kUpdSteps;
  const uint64_t tile = (uint64_t)kUpdThreads * 4 * groups * steps;
  for (size_t i = 0; i < n; i++) {
    const pots_update_weight& w = weights[i];
    // an empty weight may come with null data pointers
    if ((w.n && (!w.w_t || !w.w_next)) || w.n_parts < 1 || w.n_parts > POTS_UPDATE_MAX_PARTS)
      return POTS_E_ARG;
    UpdJob& J = jobs[i];
    memset(&J, 0, sizeof J);
    J.w_t = reinterpret_cast<uint64_t>(w.w_t);
    J.w_next = reinterpret_cast<uint64_t>(w.w_next);
    J.n_parts = w.n_parts;
    for (uint32_t p = 0; p < w.n_parts; p++) {
      if ((w.n && !w.parts[p]) || w.part_dtype[p] > 1) return POTS_E_ARG;
      J.parts[p] = reinterpret_cast<uint64_t>(w.parts[p]);
      J.part_dt[p] = w.part_dtype[p];
      bytes += w.n * (w.part_dtype[p] == 1 ? 2 : 4);
    }
    J.n = w.n;
    J.tau_w = w.tau_w;
    bool aligned = (J.w_t % 16 == 0) && (J.w_next % 16 == 0);
    for (uint32_t p = 0; p < w.n_parts; p++) aligned = aligned && J.parts[p] % 16 == 0;
    J.vec = aligned ? 1 : 0;
    J.block_first = blk.size();
    const uint64_t nb = (w.n + tile - 1) / tile;
    if (blk.size() + nb >= 0x7FFFFFFFull) return POTS_E_ARG;
    blk.insert(blk.end(), nb, (uint32_t)i);
    bytes += 8 * w.n;
  }
  UpdatePlan* P = new (std::nothrow) UpdatePlan;
  if (!P) return POTS_E_NOMEM;
  P->n = n;
  P->eta = eta;
  P->eps_w = eps_w;
  P->groups = groups;
  P->steps = steps;
  P->n_blocks = (uint32_t)blk.size();
  P->bytes = bytes;
  const size_t o_blk = align_up(n * sizeof(UpdJob), 256);
  const size_t total = o_blk + std::max<size_t>(blk.size(), 1) * 4;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&P->base), total);
  if (e != hipSuccess) {
    note_hip_error(e, "hipMalloc(update plan)", __FILE__, __LINE__);
    delete P;
    return e == hipErrorOutOfMemory ? POTS_E_NOMEM : POTS_E_HIP;
  }
  P->d_jobs = reinterpret_cast<UpdJob*>(P->base);
  P->d_blk = reinterpret_cast<uint32_t*>(P->base + o_blk);
  e = hipMemcpy(P->d_jobs, jobs.data(), n * sizeof(UpdJob), hipMemcpyHostToDevice);
  if (e == hipSuccess && !blk.empty())
    e = hipMemcpy(P->d_blk, blk.data(), blk.size() * 4, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    note_hip_error(e, "hipMemcpy(update plan)", __FILE__, __LINE__);
    (void)hipFree(P->base);
    delete P;
    return POTS_E_HIP;
  }
  *plan = P;
  return POTS_E_OK;
}

extern "C" int pots_update_plan_run(void* plan, pots_update_result* d_out, void* stream) {
  UpdatePlan* P = static_cast<UpdatePlan*>(plan);
  if (!P || !d_out) return POTS_E_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  UpdOut* out = reinterpret_cast<UpdOut*>(d_out);
  hipLaunchKernelGGL(update_init, dim3((uint32_t)((P->n + kUpdThreads - 1) / kUpdThreads)),
                     dim3(kUpdThreads), 0, s, out, (uint32_t)P->n);
  POTS_HIP(hipGetLastError());
  if (P->n_blocks) {
    const auto kernel = P->groups == 1  ? update_kernel<1, 1>
                        : P->steps == 1 ? update_kernel<kUpdGroups, 1>
                                        : update_kernel<kUpdGroups, kUpdSteps>;
    hipLaunchKernelGGL(kernel, dim3(P->n_blocks), dim3(kUpdThreads), 0, s, P->d_jobs, P->d_blk,
                       P->eta, P->eps_w, out);
    POTS_HIP(hipGetLastError());
  }
  return POTS_E_OK;
}

extern "C" uint64_t pots_update_plan_bytes(void* plan) {
  UpdatePlan* P = static_cast<UpdatePlan*>(plan);
  return P ? P->bytes : 0;
}

extern "C" void pots_update_plan_destroy(void* plan) {
  UpdatePlan* P = static_cast<UpdatePlan*>(plan);
  if (!P) return;
  if (P->base) (void)hipFree(P->base);
  delete P;
}
