// attn_fwd_wide.hpp - the forward kernel without the causal mask at head_dim 32 and 64, for grids
// that fill the GPU: 256-row programs whose four waves hold 64 rows each, as two 32-row blocks.
//
// Same tiles, same arithmetic per row as attn_fwd_kernel.hpp (64-key tiles, the lazily moved
// reference, the rounded-P sum, the key-norm bound): the output is the same bit for bit. At these
// head dims a tile's softmax takes more issue time than its MFMAs, and the clock is held down by
// power. What changes:
//   * a wave has two row blocks to interleave: S of the second block beside the softmax of the
//     first, PV of the first beside the softmax of the second (no second S tile of the same rows
//     across a barrier, as the general kernel's pipelined loop needs);
//   * every K and V operand read from LDS feeds two MFMAs instead of one, and a tile staged from L2
//     serves 256 rows instead of 128.
// Two waves per SIMD at head_dim 64 (214-220 VGPRs), three at 32 (155-161), each of another workgroup, so
// that their phases are independent; the general kernel's 8-wave programs of 256 rows share a barrier instead, and lose.
// Measured on MI355X against the general kernel (us, same box): fp16 full B2 H16 N16384 D64 at half
// scale (key-norm table) 2198.5 -> 2078.3, bf16 2088.8 -> 1994.8; B8 H16 N2048 D64 162.5 -> 155.4;
// D32 164.3 -> 156.8 (fp16 B12 N2048). Causal programs of 256 rows lose what this gains to their coarser
// tail (D64 B4 H16 N4096 162.6 -> 163.2, B2 86.4 -> 95.2), so there is no causal instance.
#pragma once

#include "attn_fwd_kernel.hpp"

namespace fa2 {

template <int DT, int D, bool KB>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2)))
void attn_wide_kernel(const Params p) {
  using E = Elem<DT>;
  constexpr int BN = 64, RB = 2, NW = 4;
  constexpr int KS = D / 16, DB = D / 32, NB = BN / 32, NT = BN / 16;
  static_assert((D == 32 || D == 64) && KS * NB == NT * DB);
  constexpr int CPR = D / 8, TCH = BN * CPR, NI = TCH / 64, JW = NI / NW;

  __shared__ u32x4 k_lds[2][TCH];
  __shared__ u32x4 v_lds[2][TCH];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 31;
  const int g = lane >> 5;

  const Program pr = program_of<false>(p, (int)blockIdx.x);

  // ---- this lane's rows, one of each row block (attn_fwd_kernel's row mapping)
  bool row_ok[RB];
  u32x4 qreg[RB][KS];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = pr.tile * p.block_m + wave * 64 + rb * 32 + c;
    const int pos = r / p.pack;
    const int head = pr.hq0 + (r - pos * p.pack);
    row_ok[rb] = pos < p.n_q;
    const uint16_t* qrow = p.q + pr.b * p.sqb + head * p.sqh + (int64_t)pos * p.sqn + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qreg[rb][ks] = row_ok[rb] ? *(const u32x4*)(qrow + 16 * ks) : u32x4{0u, 0u, 0u, 0u};
  }

  const int full_end = (p.n_kv / BN) * BN;  // tiles past it need the key mask
  const int n_tiles = (p.n_kv + BN - 1) / BN;

  // ---- score bound from the key-norm table (attn_fwd_kernel.hpp)
  float km = 0.f;
  if (KB) {
    const float* kn = p.key_norm2 + (int64_t)(pr.b * (p.h_q / p.group) + pr.hkv) * p.key_chunks;
    for (int x = lane; x < p.key_chunks; x += 64) km = fmaxf(km, kn[x]);
  }
  bool skip_row[RB] = {false, false};
  bool skip_max = false;

  // ---- K/V staging (attn_fwd_kernel.hpp)
  const char* kbase = (const char*)(p.k + pr.b * p.skb + pr.hkv * p.skh);
  const char* vbase = (const char*)(p.v + pr.b * p.svb + pr.hkv * p.svh);
  uint32_t koff[JW], voff[JW];
#pragma unroll
  for (int jj = 0; jj < JW; ++jj) {
    const int P = (wave + jj * NW) * 64 + lane;
    const int row = P / CPR, col = P % CPR;
    koff[jj] = (uint32_t)(row * p.skn + (col ^ k_key<D>(pi_row(row & 31) & 15)) * 8) * 2u;
    voff[jj] = (uint32_t)(row * p.svn + (col ^ v_key<D>(row & 15)) * 8) * 2u;
  }
  auto rsrc_at = [&](const char* base, int64_t stride, int n0) {
    const uint32_t stride2 = (uint32_t)stride * 2u;
    const uint32_t rows = (uint32_t)min(p.n_kv - n0, BN);
    return make_desc(base + (uint64_t)(uint32_t)n0 * stride2, (rows - 1u) * stride2 + (uint32_t)D * 2u);
  };
  auto issue_k = [&](int j) {
    const auto rs = rsrc_at(kbase, p.skn, j * BN);
#pragma unroll
    for (int jj = 0; jj < JW; ++jj)
      load_lds16(rs, koff[jj], lds_addr((const FA2_LDS char*)k_lds[j & 1] + (wave + jj * NW) * 1024));
  };
  auto issue_v = [&](int j) {
    const auto rs = rsrc_at(vbase, p.svn, j * BN);
#pragma unroll
    for (int jj = 0; jj < JW; ++jj)
      load_lds16(rs, voff[jj], lds_addr((const FA2_LDS char*)v_lds[j & 1] + (wave + jj * NW) * 1024));
  };

  // ---- LDS operand reads (attn_fwd_kernel.hpp)
  const int kk = k_key<D>(c & 15);
  const int vj = (lane & 15) >> 2;
  const int vq = lane & 3;
  const int vsig = ((vq & 1) << 1) | ((vq & 2) >> 1);
  const int vdh = (lane >> 4) & 1;
  uint32_t koffs[KS], voffs[2][DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koffs[ks] = (uint32_t)((pi_row(c) * CPR + ((2 * ks + g) ^ kk)) * 16);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(koffs[ks]));
#pragma unroll
  for (int rr = 0; rr < 2; ++rr)
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int row = 8 * g + 4 * rr + vj;
      const int chunk = (4 * db + 2 * vdh + (vsig >> 1)) ^ v_key<D>(row);
      voffs[rr][db] = (uint32_t)(row * (D * 2) + chunk * 16 + (vsig & 1) * 8);
    }
  auto k_operand = [&](int j, int ks, int nb) {
    return *(const u32x4 FA2_LDS*)((const char FA2_LDS*)k_lds[j & 1] + koffs[ks] + nb * 32 * CPR * 16);
  };
  auto v_operand = [&](int j, int t, int db) {
    const char FA2_LDS* vt = (const char FA2_LDS*)v_lds[j & 1];
    const u32x2 lo = lds_read_tr(vt + voffs[0][db] + t * 16 * D * 2);
    const u32x2 hi = lds_read_tr(vt + voffs[1][db] + t * 16 * D * 2);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };

  float m_i[RB] = {-INFINITY, -INFINITY}, l_i[RB] = {0.f, 0.f}, l_exact[RB] = {0.f, 0.f};
  const bool want_exact = p.lse != nullptr;
  f32x16 acc[RB][DB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[rb][db] = f32x16{};
  const float qk_scale = p.qk_scale;

  issue_k(0);
  issue_v(0);
  if (n_tiles > 1) issue_k(1);
  if (n_tiles > 1) wait_vmcnt<2 * JW>();
  else wait_vmcnt<JW>();
  __syncthreads();
  u32x4 kop[KS][NB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      kop[ks][nb] = *(const volatile u32x4 FA2_LDS*)((const char FA2_LDS*)k_lds[0] + koffs[ks] + nb * 32 * CPR * 16);
  float bound[RB] = {INFINITY, INFINITY};
  if (KB) {
#pragma unroll
    for (int off = 32; off >= 1; off /= 2) km = fmaxf(km, __shfl_xor(km, off, 64));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float qn = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int w = 0; w < 4; ++w) qn = E::sumsq2(qreg[rb][ks][w], qn);
      bound[rb] = __builtin_sqrtf(pair_sum(qn) * km) * qk_scale_bound(qk_scale);
    }
  }

  auto mask_max = [&](f32x16 (&s)[NB], int rb, int j) {
    const int n0 = j * BN;
    if (n0 + BN > full_end) {
      const int lim = p.n_kv - 1 - n0 - 8 * g;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (nb * 32 + 16 * (i / 8) + (i % 8) > lim) s[nb][i] = -INFINITY;
    }
    if (!KB || !skip_max) {
      float mx = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[nb][i]);
      mx = pair_max(mx) * qk_scale;
      const bool grow = !skip_row[rb] && mx > m_i[rb] + kRescaleTau;
      if (__builtin_amdgcn_ballot_w64(grow)) {
        const float m_new = grow ? mx : m_i[rb];
        const float alpha = __builtin_amdgcn_exp2f(m_i[rb] - m_new);
        l_i[rb] *= alpha;
        l_exact[rb] *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[rb][db] *= alpha;
        m_i[rb] = m_new;
      }
      if (KB && j == 0) {
        const float lift = bound[rb] <= kBoundLiftMax<DT> ? kBoundLift<DT> : 0.f;
        skip_row[rb] = bound[rb] <= m_i[rb] + (kBoundTau<DT> + lift);
        if (skip_row[rb]) m_i[rb] += fmaxf(0.f, ceilf(bound[rb] - kBoundTau<DT> - m_i[rb]));
      }
    }
  };
  auto softmax_p = [&](f32x16 (&s)[NB], int rb, u32x4 (&pb)[NT]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        s[nb][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[nb][i], qk_scale, -m_i[rb]));
    float rs0 = 0.f, rs1 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int nb = t >> 1, h = t & 1;
      pb[t] = u32x4{E::pack2(s[nb][8 * h + 0], s[nb][8 * h + 1]), E::pack2(s[nb][8 * h + 2], s[nb][8 * h + 3]),
                    E::pack2(s[nb][8 * h + 4], s[nb][8 * h + 5]), E::pack2(s[nb][8 * h + 6], s[nb][8 * h + 7])};
      rs0 = E::sum2(pb[t][0], rs0);
      rs1 = E::sum2(pb[t][1], rs1);
      rs0 = E::sum2(pb[t][2], rs0);
      rs1 = E::sum2(pb[t][3], rs1);
    }
    l_i[rb] += rs0 + rs1;
  };
  // Vector and exp instructions placed after each MFMA of a block: 4 + 4; 6 to 12 vector and 1 to 4
  // exp instructions measured within 1% of it, 10 + 4 2-4% slower at head_dim 64.
  constexpr int kVpm = 4, kEpm = 4;
  for (int j = 0; j < n_tiles; ++j) {
    wait_vmcnt<0>();  // V_j and K_{j+1} (this wave's part)
    __syncthreads();  // ... every wave's; every wave has read K_j's operands and is done with V_{j-1}
    if (j + 2 < n_tiles) issue_k(j + 2);
    if (j + 1 < n_tiles) issue_v(j + 1);
    f32x16 s0[NB], s1[NB];
    u32x4 pb0[NT], pb1[NT];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) s0[nb] = s1[nb] = f32x16{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) s0[nb] = E::mma(kop[ks][nb], qreg[0][ks], s0[nb]);
    mask_max(s0, 0, j);
    // block: S1's MFMAs beside softmax 0
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) s1[nb] = E::mma(kop[ks][nb], qreg[1][ks], s1[nb]);
    softmax_p(s0, 0, pb0);
#pragma unroll
    for (int x = 0; x < KS * NB; ++x) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, kVpm, 0);
      __builtin_amdgcn_sched_group_barrier(0x400, kEpm, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" ::"v"(pb0[t]));
    asm volatile("" ::"v"(l_i[0]));
    if (want_exact) l_exact[0] += lane_sum(s0);
    u32x4 va[NT][DB];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int db = 0; db < DB; ++db) va[t][db] = v_operand(j, t, db);
    mask_max(s1, 1, j);
    if (KB && j == 0) skip_max = __builtin_amdgcn_ballot_w64(!(skip_row[0] && skip_row[1])) == 0;
    // block: PV0 beside softmax 1
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int db = 0; db < DB; ++db) acc[0][db] = E::mma(va[t][db], pb0[t], acc[0][db]);
    softmax_p(s1, 1, pb1);
#pragma unroll
    for (int x = 0; x < NT * DB; ++x) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, kVpm, 0);
      __builtin_amdgcn_sched_group_barrier(0x400, kEpm, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" ::"v"(pb1[t]));
    asm volatile("" ::"v"(l_i[1]));
    if (want_exact) l_exact[1] += lane_sum(s1);
    // PV1, with K_{j+1}'s operands read beside it (a harmless stale read after the last tile)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        acc[1][db] = E::mma(va[t][db], pb1[t], acc[1][db]);
        const int y = t * DB + db;
        kop[y / NB][y % NB] = k_operand(j + 1, y / NB, y % NB);
      }
  }
  // ---- normalise once, store once
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const float l = pair_sum(l_i[rb]);
    const float lx = want_exact ? pair_sum(l_exact[rb]) : l;
    const float inv_l = 1.0f / l;
    if (!row_ok[rb]) continue;
    const int r = pr.tile * p.block_m + wave * 64 + rb * 32 + c;
    const int pos = r / p.pack;
    const int head = pr.hq0 + (r - pos * p.pack);
    uint16_t* orow = p.o + pr.b * p.sob + head * p.soh + (int64_t)pos * p.son;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x16& a = acc[rb][db];
        *(u32x4*)(orow + 32 * db + 16 * h + 8 * g) =
            u32x4{E::pack2(a[8 * h + 0] * inv_l, a[8 * h + 1] * inv_l),
                  E::pack2(a[8 * h + 2] * inv_l, a[8 * h + 3] * inv_l),
                  E::pack2(a[8 * h + 4] * inv_l, a[8 * h + 5] * inv_l),
                  E::pack2(a[8 * h + 6] * inv_l, a[8 * h + 7] * inv_l)};
      }
    if (p.lse && g == 0)
      p.lse[((int64_t)pr.b * p.h_q + head) * p.n_q + pos] = (m_i[rb] + log2f(lx)) * kLn2;
  }
}

}  // namespace fa2
