// gemm_device.h — what the matmul kernels (matmul.hip, gemm_pipe.hip) share: their launch
// parameters, the GEMMs' work order, epilogue and barrier.
#pragma once
#include "sv_device.h"
#include "sv_internal.h"

namespace sv {

struct MMParams {
  const uint8_t* w;
  const uint16_t* scales;
  const float* x;
  const uint32_t* x_rows;
  float* y;
  const float* base;
  float* aux;
  uint32_t n, k, m, epi, flags, vocab_real, gshift, chunks, per_row, tiled;
  float scale, ra, rb;
  // Split-k hand-off (skinny path with S > 1): counters per row group (zero at rest),
  // partial sums and sums of squares per (row group, split).
  uint32_t* counters;
  float* part;
  float* ssp;
  uint32_t splits, tgroups;  // skinny: k splits and 16-token groups
  // GEMM work order (gemm_item): 0 row block, split, token block (token block fastest); g > 0:
  // split, groups of g row blocks, token block, row block within the group.
  uint32_t order;
};

// The GEMMs' work item -> (token block, split, row block). Each XCD (workgroup id mod 8) takes a
// contiguous range of items, so the order decides which weights (row block, split) and which
// activations (token block, split) one XCD's L2 serves to several workgroups; the host picks the
// order with the least modelled HBM traffic (gemm_order).
__device__ __forceinline__ void gemm_item(uint32_t item, uint32_t n_tblk, uint32_t S, uint32_t nrb, uint32_t g,
                                          uint32_t& tblk, uint32_t& sp, uint32_t& rblk) {
  if (g == 0) {
    tblk = item % n_tblk;
    sp = (item / n_tblk) % S;
    rblk = item / (n_tblk * S);
    return;
  }
  const uint32_t per_sp = nrb * n_tblk, per_grp = g * n_tblk;
  sp = item / per_sp;
  const uint32_t rem = item % per_sp, r2 = rem % per_grp;
  tblk = r2 / g;
  rblk = (rem / per_grp) * g + r2 % g;
}


__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + __expf(-x)); }

constexpr int GKC = 64;
// Split-k hand-off counters (skinny and GEMM paths): a region of fixed size at the front of the
// workspace, so every matmul sharing one workspace finds its counters at zero there, whatever
// its shape.
constexpr size_t COUNTER_SLOTS = 65536;

// Wait for this thread's LDS operations, then the workgroup barrier. Unlike __syncthreads()
// this leaves global loads in flight (no vmcnt wait).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Epilogue of the GEMM (kernels.metal:183-209) for one 16-token tile: lane (t16, q) holds rows
// 4 q + 0..3 of each of the wave's RTW row tiles (first row row0) for token t.
template <int RTW>
__device__ __forceinline__ void gemm_epilogue(const MMParams& p, const f32x4 (&acc)[RTW], uint32_t row0, int q,
                                              uint32_t t, float ss, bool write_inv) {
  const float inv = 1.0f / __builtin_sqrtf(ss / (float)p.k + SV_RMS_EPS);
  if (write_inv && (p.flags & SV_FLAG_WRITE_INV) && p.epi == SV_EPI_NORM && q == 0) p.aux[t] = inv;
  const bool norm_in = (p.flags & SV_FLAG_NORM_IN) != 0;
#pragma unroll
  for (int r = 0; r < RTW; r++) {
    const uint32_t rowq = row0 + 16 * r + 4 * q;
    f32x4 v = acc[r];
    const size_t o = (size_t)t * p.m + rowq;
    switch (p.epi) {
      case SV_EPI_NORM:
        *(f32x4*)(p.y + o) = v * (inv * p.scale);
        break;
      case SV_EPI_RAW:
        if (norm_in) v *= inv;
        *(f32x4*)(p.y + o) = v;
        break;
      case SV_EPI_RESID: {
        if (norm_in) v *= inv;
        const f32x4 sv = v * p.scale;
        const f32x4 b = *(const f32x4*)(p.base + o);
        *(f32x4*)(p.y + o) = b * p.ra + sv * p.rb;
        if (p.flags & SV_FLAG_WRITE_RAW) *(f32x4*)(p.aux + o) = sv;
        break;
      }
      case SV_EPI_HEAD: {
        if (norm_in) v *= inv;
        f32x4 l;
#pragma unroll
        for (int i = 0; i < 4; i++)
          l[i] = rowq + i < p.vocab_real ? 23.0f * sigmoidf_((v[i] + 5.0f) / 7.5f) : -__builtin_inff();
        *(f32x4*)(p.y + o) = l;
        break;
      }
      case SV_EPI_SWIGLU: {
        const float sc = inv * p.scale;
        const float g0 = v[0] * sc, u0 = v[1] * sc, g1 = v[2] * sc, u1 = v[3] * sc;
        float2 out;
        out.x = g0 * sigmoidf_(g0) * u0;
        out.y = g1 * sigmoidf_(g1) * u1;
        *(float2*)(p.y + (size_t)t * (p.m / 2) + rowq / 2) = out;
        break;
      }
      default:
        break;
    }
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// gemm_pipe.hip: whether mm_pipe is built for this shape (32-row tiles per wave rt, 32-token
// tiles nt, chunks per iteration cpi), and its launch over nwg workgroups of 8 waves.
bool gemm_pipe_built(bool grouped, int rt, int nt, int cpi);
void gemm_pipe_launch(hipStream_t stream, uint32_t fmt, bool grouped, int rt, int nt, int cpi, const MMParams& p,
                      uint32_t nwg, uint32_t n_tblk);

}  // namespace sv
