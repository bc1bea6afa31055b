// KZG polynomial commitment over G1 for gfx950 (reference KZGCommitment,
// src/prover/groth16.cuh:188-207, groth16.cu:393-438):
//   commit(f)  = sum_i f_i [tau^i]_1                      (one G1 MSM)
//   open(f, z) = sum_i q_i [tau^i]_1,  q = (f - f(z)) / (x - z)
// with f given by its d coefficients (ascending) and q by synthetic division
//   q_{d-2} = f_{d-1},  q_i = f_{i+1} + z q_{i+1},
// i.e. q_i = sum_{j >= i} f_{j+1} z^(j-i): a suffix Horner scan, which the
// reference runs as a serial host loop.  Here it runs on the GPU as a blocked
// scan: a block folds KZG_B values (four per thread from the top, then a suffix
// scan of the threads' values in LDS), the blocks' values are scanned the same way
// with multiplier z^KZG_B (recursively, until one block is left), and a last pass
// adds z^(e-i) * q_e (q_e = scanned value of the next block) to every value.
// The map is linear, so it runs on the reference's Montgomery words
// directly (repack only) with z prepared in the internal radix.
//
// Bound by the chain of dependent products at these sizes: 12 per level here, two
// levels up to 2^20 coefficients.  Threads folding 32 values each were chains of 32
// over four levels at degree 100,000, on 49 waves in the first one, after a copy of
// the coefficients: an opening took 629 us, 534 with this and f(z) read at the end.
#include <string.h>

#include "zk_internal.hpp"

namespace zk {

constexpr int KZG_THREADS = 256;
constexpr int KZG_LOG_T = 8;
constexpr int KZG_E = 4;                    // values per thread
constexpr int KZG_B = KZG_E * KZG_THREADS;  // values per block

struct ZPow {
  fr p[KZG_E + 1];     // p[k] = y^k in the internal radix
  fr step[KZG_LOG_T];  // step[d] = y^(E 2^d)
};

__device__ __forceinline__ fr kzg_load(const uint4* __restrict__ p, size_t i) {
  uint4 a = p[2 * i], b = p[2 * i + 1];
  uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  return repack_in<FrP>(w);
}

__device__ __forceinline__ void kzg_store(uint4* __restrict__ p, size_t i, const fr& x) {
  uint32_t w[8];
  repack_out(x, w);
  p[2 * i] = make_uint4(w[0], w[1], w[2], w[3]);
  p[2 * i + 1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// Block b = [b B, min(n, (b + 1) B)): x_i = sum_{i <= j < e} in_j y^(j-i), e the
// block's end; tot[b] = the value at its start.  `in` may be x.
__global__ __launch_bounds__(KZG_THREADS) void k_kzg_fold(const uint4* in, uint4* x, size_t n, ZPow y,
                                                          uint4* __restrict__ tot) {
  __shared__ uint32_t S[2][NL][KZG_THREADS];
  const uint32_t t = threadIdx.x;
  const size_t i0 = blockIdx.x * (size_t)KZG_B + (size_t)t * KZG_E;
  fr v[KZG_E];
#pragma unroll
  for (int k = 0; k < KZG_E; k++) v[k] = i0 + k < n ? kzg_load(in, i0 + k) : fe_zero<FrP>();
#pragma unroll
  for (int k = KZG_E - 2; k >= 0; k--) v[k] = fadd(v[k], fmul(v[k + 1], y.p[1]));
  // a = the sum from this thread's first value over the next 2^d threads; two
  // buffers, so a step's writes wait for no reader of the step before
  fr a = v[0], o;
#pragma unroll 1
  for (int d = 0; d <= KZG_LOG_T; d++) {
    uint32_t(*buf)[KZG_THREADS] = S[d & 1];
#pragma unroll
    for (int l = 0; l < NL; l++) buf[l][t] = a.l[l];
    __syncthreads();
    const uint32_t off = d < KZG_LOG_T ? 1u << d : 1u;
    const bool has = t + off < KZG_THREADS;
#pragma unroll
    for (int l = 0; l < NL; l++) o.l[l] = has ? buf[l][t + off] : 0u;
    if (d < KZG_LOG_T) a = fadd(a, fmul(o, y.step[d]));
  }
  // o = the next thread's sum to the block's end
#pragma unroll
  for (int k = 0; k < KZG_E; k++) {
    if (i0 + k < n) kzg_store(x, i0 + k, fadd(v[k], fmul(o, y.p[KZG_E - k])));
  }
  if (t == 0) kzg_store(tot, blockIdx.x, a);
}

// x_i += y^(e-i) * tot[b + 1] for i in block b, e its end (tot holds the scanned
// block starts; the last block has no carry and is not launched).
__global__ __launch_bounds__(KZG_THREADS) void k_kzg_carry(uint4* __restrict__ x, ZPow y,
                                                           const uint4* __restrict__ tot) {
  const uint32_t t = threadIdx.x, back = KZG_THREADS - 1 - t;
  const size_t i0 = blockIdx.x * (size_t)KZG_B + (size_t)t * KZG_E;
  fr c = kzg_load(tot, blockIdx.x + (size_t)1);  // times y^(E back)
#pragma unroll 1
  for (int d = 0; d < KZG_LOG_T; d++) {
    const fr m = fmul(c, y.step[d]);
#pragma unroll
    for (int l = 0; l < NL; l++) c.l[l] = (back >> d) & 1u ? m.l[l] : c.l[l];
  }
#pragma unroll
  for (int k = 0; k < KZG_E; k++) kzg_store(x, i0 + k, fadd(kzg_load(x, i0 + k), fmul(c, y.p[KZG_E - k])));
}

static ZPow zpow_table(const fr& y) {
  ZPow t;
  t.p[0] = fe_one<FrP>();
  for (int k = 1; k <= KZG_E; k++) t.p[k] = fmul(t.p[k - 1], y);
  t.step[0] = t.p[KZG_E];
  for (int d = 1; d < KZG_LOG_T; d++) t.step[d] = fmul(t.step[d - 1], t.step[d - 1]);
  return t;
}

// Suffix Horner scan of n raw Montgomery elements `in` with multiplier y (internal
// radix) into x (which may be `in`); tot: scratch of tot_capacity(n) elements.
static int suffix_horner(zk_context* ctx, const uint4* in, uint4* x, size_t n, const fr& y, uint4* tot,
                         hipStream_t st) {
  if (n == 0) return ZK_OK;
  const ZPow yp = zpow_table(y);
  const size_t m = (n + KZG_B - 1) / KZG_B;
  ZK_LAUNCH(ctx, st, "kzg_division", k_kzg_fold, dim3((uint32_t)m), dim3(KZG_THREADS), 0, in, x, n, yp, tot);
  if (m == 1) return ZK_OK;  // one block: the fold is the whole scan
  const fr& top = yp.step[KZG_LOG_T - 1];
  ZK_TRY(suffix_horner(ctx, tot, tot, m, fmul(top, top), tot + 2 * m, st));
  ZK_LAUNCH(ctx, st, "kzg_division", k_kzg_carry, dim3((uint32_t)m - 1), dim3(KZG_THREADS), 0, x, yp, tot);
  return ZK_OK;
}

static size_t tot_capacity(size_t n) {
  size_t t = 0;
  do {
    n = (n + KZG_B - 1) / KZG_B;
    t += n;
  } while (n > 1);
  return t;
}

// Whether the fold may read [p, p + bytes) in place: one device allocation of
// this context's GPU that is known to hold all of it, at an address its 16-byte
// loads take.  (About a microsecond on the host; a copy of the coefficients is a
// launch and a pass over them.)
static bool readable_in_place(const zk_context* ctx, const void* p, size_t bytes) {
  if ((uintptr_t)p % 16) return false;
  hipPointerAttribute_t at;
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  const bool known = hipPointerGetAttributes(&at, p) == hipSuccess && at.type == hipMemoryTypeDevice &&
                     at.device == ctx->device &&
                     hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) == hipSuccess;
  (void)hipGetLastError();  // an address the runtime does not know is an answer, not this call's failure
  if (!known) return false;
  const size_t off = (size_t)((const uint8_t*)p - (const uint8_t*)base);
  return off <= size && bytes <= size - off;
}

static fr fr_internal(const uint64_t mont[4]) {
  uint32_t w[8];
  memcpy(w, mont, 32);
  return from_mont256<FrP>(w);
}

}  // namespace zk

extern "C" {

static int zk_kzg_commit_impl(zk_context* ctx, const void* d_srs_g1, const void* d_coeffs, size_t degree,
                              void* h_commitment, void* stream) {
  if (!ctx || !h_commitment || (degree && (!d_srs_g1 || !d_coeffs))) return ZK_ERR_INVALID;
  return zk::msm_g1_run(ctx, d_srs_g1, d_coeffs, degree, (uint64_t*)h_commitment, ctx->s(stream));
}

int zk_kzg_commit(zk_context* ctx, const void* d_srs_g1, const void* d_coeffs, size_t degree, void* h_commitment,
                  void* stream) {
  return zk::guard(ctx, [&] { return zk_kzg_commit_impl(ctx, d_srs_g1, d_coeffs, degree, h_commitment, stream); });
}

static int zk_kzg_open_impl(zk_context* ctx, const void* d_srs_g1, const void* d_coeffs, size_t degree,
                            const uint64_t z[4], void* h_proof, uint64_t f_z[4], void* stream) {
  using namespace zk;
  if (!ctx || !h_proof || !z || (degree && (!d_srs_g1 || !d_coeffs))) return ZK_ERR_INVALID;
  if (degree > MSM_MAX_N + 1) return ctx->fail(ZK_ERR_SIZE, "kzg: degree above the MSM limit");
  hipStream_t st = ctx->s(stream);
  if (degree <= 1) {  // constant polynomial: the proof is the identity (groth16.cu:414-416)
    memset(h_proof, 0, 64);
    if (f_z) {
      memset(f_z, 0, 32);
      if (degree == 1) ZK_HIP(ctx, hipMemcpyAsync(f_z, d_coeffs, 32, hipMemcpyDeviceToHost, st));
      ZK_HIP(ctx, hipStreamSynchronize(st));
    }
    return ZK_OK;
  }
  const size_t nq = degree - 1;
  const fr zi = fr_internal(z);  // read before anything is written: z may lie in h_proof or f_z
  ZK_TRY(ctx->ensure(ctx->scratch_b, nq * 32));
  ZK_TRY(ctx->ensure(ctx->scratch_c, tot_capacity(nq) * 32 + 64));
  uint4* q = (uint4*)ctx->scratch_b.p;
  // f_1 .. f_{d-1}: read in place, or as the runtime's copy takes them (other
  // memory than this GPU's, other alignments) or refuses them (a buffer too short)
  const uint4* f1 = (const uint4*)d_coeffs + 2;
  if (!readable_in_place(ctx, d_coeffs, degree * 32)) {
    ZK_HIP(ctx, hipMemcpyAsync(q, (const uint8_t*)d_coeffs + 32, nq * 32, hipMemcpyDeviceToDevice, st));
    f1 = q;
  }
  ZK_TRY(suffix_horner(ctx, f1, q, nq, zi, (uint4*)ctx->scratch_c.p, st));
  if (f_z) {
    // to pinned memory, read after the MSM has waited for the stream: a copy to
    // pageable memory and a wait of its own held the MSM's launches back
    if (!ctx->h_words) ZK_HIP(ctx, hipHostMalloc((void**)&ctx->h_words, 64, hipHostMallocDefault));
    ZK_HIP(ctx, hipMemcpyAsync(ctx->h_words, d_coeffs, 32, hipMemcpyDeviceToHost, st));
    ZK_HIP(ctx, hipMemcpyAsync(ctx->h_words + 4, q, 32, hipMemcpyDeviceToHost, st));
  }
  const int rc = msm_g1_run(ctx, d_srs_g1, q, nq, (uint64_t*)h_proof, st);
  if (rc != ZK_OK) {
    (void)hipStreamSynchronize(st);  // the copies above
    return rc;
  }
  if (f_z) {  // f(z) = f_0 + z q_0 (host, reference words)
    uint32_t a[8], b[8], out[8];
    memcpy(a, ctx->h_words, 32);
    memcpy(b, ctx->h_words + 4, 32);
    repack_out(fadd(repack_in<FrP>(a), fmul(repack_in<FrP>(b), zi)), out);
    memcpy(f_z, out, 32);
  }
  return ZK_OK;
}

int zk_kzg_open(zk_context* ctx, const void* d_srs_g1, const void* d_coeffs, size_t degree, const uint64_t z[4],
                void* h_proof, uint64_t f_z[4], void* stream) {
  return zk::guard(ctx, [&] { return zk_kzg_open_impl(ctx, d_srs_g1, d_coeffs, degree, z, h_proof, f_z, stream); });
}

}  // extern "C"
