// gemm_pipe.hip — the GEMM whose two waves per SIMD run half an iteration apart.
#include "gemm_device.h"

namespace sv {

// The GEMM for the rows that fill 32 x 32 tiles (matmul.hip pick_by_time): 8 waves, BM = 256 RT
// output rows (RT 32-row tiles per wave), BN = 32 NT tokens, 1/S of k; iterations of CPI chunks of
// 64 k. Operands and layouts are mm_gemm32's (weights straight to registers in MFMA lane order
// and converted there, X split once per workgroup to bf16 hi + lo in LDS). What differs:
//   - A SIMD's two waves alternate. Waves 0-3 prepare an iteration (weights to bf16, their half of
//     the X tile split into LDS, the loads D iterations ahead) while waves 4-7 multiply theirs,
//     then they swap, with a barrier between the half iterations: the matrix cores always have
//     one wave's products while the VALU has the other's conversions. (With all waves in one
//     phase the two added up: 4900 cycles an iteration of 512 x 64 against 2480, of which 2048
//     are the products' own; measured with the shader clock.) Group 0 writes its half of
//     iteration it's X tile, group 1 of it + 1's, so two X buffers are enough.
//   - Each step's two B operands (hi, lo) are read AHEAD steps before their products.
//   - 16 lanes read one token's 256 bytes of a chunk (whole cache lines), and a half-wave's LDS
//     writes fall on 16 different slots.
//   - Scale groups (GR, 64 k or more): a chunk's products go to a set of sums of their own, which is
//     scaled into the accumulators while the next tile's products run; a chunk's scales, one row
//     per lane, pass through the wave's own LDS words.
// What bounds it now: at 1000 rows and more the clock, not the schedule: with random operands the
// chip holds about 1.7 GHz (products alone reach 1.6-1.9 PFLOP/s of the 2.5 they reach on zeros).
// MI355X, hi + lo counted, both sides timed in turn with the weights cold: gate_up (16384 x 2048) at
// 2048 rows 219 us, 1.26 PFLOP/s (blocks of 512 x 64 with all waves in one phase: 252, 1.09); down
// (2048 x 8192) 129 us (155, blocks of 256 x 32); the two together 348 (407). The 1280-wide model's
// gate_up in groups of 64 at 2048 rows 93 us (mm_gemm: 190). Below 300 rows the operands' way from L2
// (a 256-row block reads X at 4 bytes a value), the pipeline's fill and the split's merge are as large.
template <int FMT, int RT, int NT, int CPI, bool GR>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mm_pipe(MMParams p, uint32_t n_tblk) {
  constexpr int BN = 32 * NT, D = RT * NT >= 8 ? 1 : 2;
  constexpr int ESZ = FMT == SV_FMT_I8 ? 1 : 2;
  constexpr int WL = FMT == SV_FMT_I8 ? 1 : 2;  // 16-byte words per lane per 16 k
  constexpr int UPT = NT * CPI;                 // units (4 k of one token) per thread and iteration
  __shared__ u32x4 xs[2][CPI][NT][2][256];
  __shared__ float ssp[BN][16];
  __shared__ float scl[GR ? 8 : 1][GR ? CPI : 1][GR ? 32 * RT : 1];
  __shared__ uint32_t last_flag;
  const int tid = threadIdx.x, lane = tid & 63, c32 = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t grp = wv >> 2;  // waves 0-3 / 4-7: one of each group per SIMD

  const uint32_t nwg = gridDim.x, S = p.splits;
  const uint32_t xcd = blockIdx.x % 8, xq = nwg / 8;
  const uint32_t item = xcd * xq + min(xcd, nwg % 8) + blockIdx.x / 8;
  uint32_t tblk, sp, rblk;
  gemm_item(item, n_tblk, S, nwg / (n_tblk * S), p.order, tblk, sp, rblk);
  const uint32_t t0 = tblk * BN;
  const uint32_t row0 = (rblk * 8 + wv) * 32 * RT;  // this wave's first row
  const uint32_t nc = __builtin_amdgcn_readfirstlane(p.k / GKC / S);
  const uint32_t cb = __builtin_amdgcn_readfirstlane(sp * nc);

  const __amdgpu_buffer_rsrc_t xrs = coherent_rsrc(p.x), wrs = coherent_rsrc(p.w);
  constexpr uint32_t OOB = 0x80000000u;
  const uint32_t tile_bytes = 16 * p.k * ESZ;  // one 16-row block over all k
  const uint32_t wl = p.tiled ? (uint32_t)(c32 >> 4) * tile_bytes + (uint32_t)((c32 & 15) + 32 * h) * 16
                              : ((uint32_t)c32 * p.k + 32 * h) * ESZ;
  const uint32_t chunk_bytes = p.tiled ? 1024 * ESZ : 64 * ESZ, qq_bytes = p.tiled ? 256 : 16 * ESZ,
                 v_bytes = p.tiled ? 1024 : 16;
  // X units: 16 lanes read one token's 256 bytes of a chunk; a group of 4 waves takes 16 tokens
  // per pass, group g the passes j with token bit 4 = g, over every 32-token tile and chunk.
  // Consecutive 16-lane groups differ in token bit 3, so a half-wave's 8-byte LDS writes fall on
  // 16 different slots mod 16.
  const uint32_t kq = tid & 15, tg = (tid & 255) >> 4;
  const uint32_t tok16 = ((tg & 1) << 3) | (tg >> 1) | (grp << 4);  // 0 .. 31
  uint32_t xoff[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) {
    const uint32_t tt = t0 + 32 * n + tok16;
    xoff[n] = tt < p.n ? ((p.x_rows ? p.x_rows[tt] : tt) * p.k + 4 * kq) * 4 : OOB;
  }
  const uint32_t g8 = kq >> 1;  // 8-k group 4 h + ks
  const uint32_t xslot = (64 * (g8 & 3) + 32 * (g8 >> 2) + (tok16 ^ g8)) * 16 + 8 * (kq & 1);
  auto load_x = [&](uint32_t it, f32x4 (&xr)[UPT]) {
#pragma unroll
    for (int u = 0; u < CPI; u++) {
      const uint32_t c = it * CPI + u;
      const uint32_t so = __builtin_amdgcn_readfirstlane((cb + min(c, nc - 1)) * GKC * 4);
#pragma unroll
      for (int n = 0; n < NT; n++) xr[u * NT + n] = __builtin_bit_cast(f32x4, buf_ld16(xrs, c < nc ? xoff[n] : OOB, so));
    }
  };
  auto load_w = [&](uint32_t it, u32x4 (&wr)[CPI][RT][2 * WL]) {
#pragma unroll
    for (int u = 0; u < CPI; u++) {
      const uint32_t c = it * CPI + u, cc = c < nc ? cb + c : 0u;
      const uint32_t vo = c < nc ? wl : OOB;
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int qq = 0; qq < 2; qq++)
#pragma unroll
          for (int v = 0; v < WL; v++) {
            const uint32_t rbase = p.tiled ? (row0 / 16 + 2 * r) * tile_bytes : (row0 + 32 * r) * p.k * ESZ;
            wr[u][r][qq * WL + v] =
                buf_ld16(wrs, vo, __builtin_amdgcn_readfirstlane(rbase + cc * chunk_bytes + qq * qq_bytes + v * v_bytes));
          }
    }
  };
  // Scale groups of at least one chunk: lane l holds row l's scale of each chunk.
  const uint32_t ng = p.per_row ? 1u : p.k >> p.gshift;
  const uint16_t* srow = GR ? p.scales + (size_t)(row0 + (RT == 2 ? lane : c32)) * ng : nullptr;
  auto load_s = [&](uint32_t it, float (&sr)[CPI]) {
    if constexpr (GR)
#pragma unroll
      for (int u = 0; u < CPI; u++) sr[u] = bf(ldg_u16(srow + (((cb + min(it * CPI + u, nc - 1)) * GKC) >> p.gshift)));
  };
  float ssacc[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) ssacc[n] = 0.0f;
  auto store_x = [&](uint32_t it, const f32x4 (&xr)[UPT]) {
    char* buf = (char*)&xs[0][0][0][0][0] + (it & 1) * (CPI * NT * 8192) + xslot;
#pragma unroll
    for (int u = 0; u < CPI; u++)
#pragma unroll
      for (int n = 0; n < NT; n++) {
        const f32x4 v = xr[u * NT + n];
#pragma unroll
        for (int e = 0; e < 4; e++) ssacc[n] = __builtin_fmaf(v[e], v[e], ssacc[n]);
        const u32x2 s01 = split2(v[0], v[1]), s23 = split2(v[2], v[3]);
        *(u32x2*)(buf + (u * NT + n) * 8192) = u32x2{s01[0], s23[0]};
        *(u32x2*)(buf + (u * NT + n) * 8192 + 4096) = u32x2{s01[1], s23[1]};
      }
  };

  f32x16 acc[RT][NT];
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[r][n][e] = 0.0f;

  f32x4 xr[D][UPT];
  u32x4 wr[D][CPI][RT][2 * WL];
  float sr[D][CPI];
  {
    f32x4 x0[UPT];
    load_x(0, x0);
#pragma unroll
    for (int d = 0; d < D; d++) {
      load_w(d, wr[d]);
      load_s(d, sr[d]);
      load_x(d + grp, xr[d]);
    }
    if (grp) store_x(0, x0);
  }
  const uint32_t ni = (nc + CPI - 1) / CPI;
  if (grp) lds_barrier();

  auto body = [&](uint32_t it, int d) {
    // Prepare: this iteration's weights as bf16 operands, this group's half of the X tile
    // (group 0: iteration it's, group 1: the next one's), the loads D iterations ahead.
    store_x(it + grp, xr[d]);
    bf16x8 a[CPI][RT][4];
#pragma unroll
    for (int u = 0; u < CPI; u++)
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
          if (FMT == SV_FMT_I8) {
            const u32x4 w = wr[d][u][r][ks >> 1];
            a[u][r][ks] = i8x8_to_bf(w[2 * (ks & 1)], w[2 * (ks & 1) + 1]);
          } else {
            a[u][r][ks] = __builtin_bit_cast(bf16x8, wr[d][u][r][ks]);
          }
        }
    if constexpr (GR)
#pragma unroll
      for (int u = 0; u < CPI; u++) scl[wv][u][RT == 2 ? lane : c32] = sr[d][u];
    load_x(it + grp + D, xr[d]);
    load_w(it + D, wr[d]);
    load_s(it + D, sr[d]);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // Multiply, while the SIMD's other wave prepares. Step s (chunk, k step, token tile; with
    // scale groups chunk, token tile, k step) takes two B operands, read AHEAD steps before.
    __builtin_amdgcn_s_setprio(1);
    constexpr int STEPS = CPI * 4 * NT, AHEAD = RT * NT >= 8 ? 1 : RT == 2 ? 2 : 3, RING = AHEAD + 1;
    bf16x8 b[RING][2];
    const u32x4* xb = &xs[0][0][0][0][0] + (it & 1) * (CPI * NT * 512);
    auto step = [&](int s, int& u, int& ks, int& n) {
      u = s / (4 * NT);
      if (GR) ks = s % 4, n = s / 4 % NT;
      else ks = s / NT % 4, n = s % NT;
    };
    auto read_b = [&](int s) {
      int u, ks, n;
      step(s, u, ks, n);
      const int slot = 64 * ks + 32 * h + (c32 ^ (4 * h + ks));
#pragma unroll
      for (int hl = 0; hl < 2; hl++) b[s % RING][hl] = __builtin_bit_cast(bf16x8, xb[((u * NT + n) * 2 + hl) * 256 + slot]);
    };
#pragma unroll
    for (int s = 0; s < AHEAD; s++) read_b(s);
    f32x16 g[GR ? 2 : 1][GR ? RT : 1];
    f32x4 sc[GR ? RT : 1][4];
    auto scale = [&](int set, int n) {
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          acc[r][n][e] = __builtin_fmaf(sc[GR ? r : 0][e >> 2][e & 3], g[GR ? set : 0][GR ? r : 0][e], acc[r][n][e]);
    };
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      int u, ks, n;
      step(s, u, ks, n);
      if (s + AHEAD < STEPS) read_b(s + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (GR) {
        const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const int set = (s / 4) & 1;
#pragma unroll
        for (int hl = 0; hl < 2; hl++)
#pragma unroll
          for (int r = 0; r < RT; r++) g[set][r] = mfma32(a[u][r][ks], b[s % RING][hl], ks == 0 && hl == 0 ? zero : g[set][r]);
        // the group before this one: its products have left the matrix cores by now
        if (ks == 0 && s > 0) scale(set ^ 1, (n + NT - 1) % NT);
        if (ks == 1 && n == 0)
#pragma unroll
          for (int r = 0; r < RT; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) sc[r][j] = *(const f32x4*)&scl[wv][u][32 * r + 8 * j + 4 * h];
      } else {
#pragma unroll
        for (int hl = 0; hl < 2; hl++)
#pragma unroll
          for (int r = 0; r < RT; r++) acc[r][n] = mfma32(a[u][r][ks], b[s % RING][hl], acc[r][n]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (GR) scale((STEPS / 4 - 1) & 1, NT - 1);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  uint32_t it = 0;
  if constexpr (D == 2) {
    for (; it + 2 <= ni; it += 2) {
      body(it, 0);
      body(it + 1, 1);
    }
    if (it < ni) body(it, 0);
  } else {
    for (; it < ni; it++) body(it, 0);
  }
  if (!grp) lds_barrier();

  // Per-row int8 scales: lane (c, h) holds rows 8 j + 4 h + i of each tile.
  if (FMT == SV_FMT_I8 && !GR) {
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint16_t* sp4 = p.scales + row0 + 32 * r + 8 * j + 4 * h;  // any alignment
        const float s0 = bf(ldg_u16(sp4)), s1 = bf(ldg_u16(sp4 + 1)), s2 = bf(ldg_u16(sp4 + 2)),
                    s3 = bf(ldg_u16(sp4 + 3));
#pragma unroll
        for (int n = 0; n < NT; n++) {
          acc[r][n][4 * j + 0] *= s0;
          acc[r][n][4 * j + 1] *= s1;
          acc[r][n][4 * j + 2] *= s2;
          acc[r][n][4 * j + 3] *= s3;
        }
      }
  }
#pragma unroll
  for (int n = 0; n < NT; n++) ssp[32 * n + tok16][kq] = ssacc[n];
  __syncthreads();
  auto token_ss = [&](uint32_t tl) {
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) ss += ssp[tl][e];
    return ss;
  };
  float ssn[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) ssn[n] = token_ss(32 * n + c32);

  if (S > 1) {
    // [cell][split][512 threads][RT NT 4] f32x4 and [cell][split][BN] sums of squares; the
    // last split of the cell adds them in split order.
    const uint32_t cell = rblk * n_tblk + tblk;
    const __amdgpu_buffer_rsrc_t prs = coherent_rsrc(p.part), srs = coherent_rsrc(p.ssp);
    constexpr uint32_t PER = 512 * RT * NT * 64;
    const uint32_t pb = (cell * S) * PER;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          store_wt4(prs, pb + sp * PER + (((r * NT + n) * 4 + j) * 512 + tid) * 16,
                    f32x4{acc[r][n][4 * j], acc[r][n][4 * j + 1], acc[r][n][4 * j + 2], acc[r][n][4 * j + 3]});
    for (int tt = tid; tt < BN; tt += 512)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(token_ss(tt)), srs, ((cell * S + sp) * BN + tt) * 4, 0,
                                            SV_CPOL_SC1);
    if (!arrive_last(p.counters + cell, S, &last_flag)) return;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[r][n][e] = 0.0f;
#pragma unroll
    for (int n = 0; n < NT; n++) ssn[n] = 0.0f;
    for (uint32_t s2 = 0; s2 < S; s2++) {
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const f32x4 v = load_wt4(prs, pb + s2 * PER + (((r * NT + n) * 4 + j) * 512 + tid) * 16);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[r][n][4 * j + i] += v[i];
          }
#pragma unroll
      for (int n = 0; n < NT; n++)
        ssn[n] += __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(srs, ((cell * S + s2) * BN + 32 * n + c32) * 4, 0, SV_CPOL_SC1));
    }
  }

  // Epilogue: each (tile, token tile, j) is a group of 4 rows for token t0 + 32 n + c.
#pragma unroll
  for (int n = 0; n < NT; n++) {
    const uint32_t t = t0 + 32 * n + c32;
    if (t >= p.n) continue;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        f32x4 col[1] = {f32x4{acc[r][n][4 * j], acc[r][n][4 * j + 1], acc[r][n][4 * j + 2], acc[r][n][4 * j + 3]}};
        gemm_epilogue<1>(p, col, row0 + 32 * r + 8 * j + 4 * h, 0, t, ssn[n],
                         rblk == 0 && wv == 0 && r == 0 && j == 0 && h == 0);
      }
  }
}

// With scale groups the 512-row blocks of 64 and 128 tokens hold two sets of sums, and spill: not built.
bool gemm_pipe_built(bool grouped, int rt, int nt, int cpi) {
  return (rt == 1 && ((nt == 1 && cpi == 2) || (nt == 2 && cpi == 2) || (nt == 4 && cpi == 1))) ||
         (rt == 2 && cpi == 1 && (nt == 1 || (!grouped && (nt == 2 || nt == 4))));
}

void gemm_pipe_launch(hipStream_t stream, uint32_t fmt, bool grouped, int rt, int nt, int cpi, const MMParams& p,
                      uint32_t nwg, uint32_t n_tblk) {
#define SV_PIPE(F, R, N, C, G)                                                         \
  if (rt == R && nt == N && cpi == C) {                                                \
    launch((mm_pipe<F, R, N, C, G>), dim3(nwg), dim3(512), 0, stream, p, n_tblk);      \
    return;                                                                            \
  }
#define SV_PIPE_F(F, G) SV_PIPE(F, 1, 1, 2, G) SV_PIPE(F, 1, 2, 2, G) SV_PIPE(F, 1, 4, 1, G) SV_PIPE(F, 2, 1, 1, G)
  if (fmt != SV_FMT_I8) {
    SV_PIPE_F(SV_FMT_BF16, false) SV_PIPE(SV_FMT_BF16, 2, 2, 1, false) SV_PIPE(SV_FMT_BF16, 2, 4, 1, false)
  } else if (grouped) {
    SV_PIPE_F(SV_FMT_I8, true)
  } else {
    SV_PIPE_F(SV_FMT_I8, false) SV_PIPE(SV_FMT_I8, 2, 2, 1, false) SV_PIPE(SV_FMT_I8, 2, 4, 1, false)
  }
#undef SV_PIPE_F
#undef SV_PIPE
}

}  // namespace sv
