// attn_fwd_wavesplit.hpp - the forward kernel for launches that leave the general kernel's waves
// idle: few query rows per KV head against a long K/V (decoding, scoring a few drafted tokens),
// and grids too small to fill the GPU (short prompts, cross-attention). Same attention, same
// per-row recurrence as attn_fwd_kernel.hpp (fa2/kernel.py:60-183); what differs is who shares
// what.
//
// The general kernel gives every wave 32 rows of its own and walks all of a program's keys with
// each of them. With 1 to 32 rows per KV head three of its four waves multiply zeros; on a small
// grid a CU holds one workgroup, one wave per SIMD, and the launch takes as long as its longest
// key range (0.68-1.15 us per 64-key tile and wave, whatever the other CUs do). Here the four
// waves of a workgroup are KG key groups of GW = 4 / KG waves: a group's waves hold 32 rows each
// and share K/V tiles, and the groups take the key tiles in turn (tile t belongs to group
// t % KG), so a row's keys are walked by KG waves at once. Each group keeps its own (m, l, O);
// the groups meet once, in LDS, after the last tile.
//   * GW = 1 (32 rows, four key groups): every wave streams tiles of its own through LDS buffers
//     of its own, so the tile loop has no barrier, only waits on the wave's own loads, and each
//     buffer is refilled as soon as its operands are in registers. Bound by reading K and V where
//     rows are few.
//   * GW = 2 (64 rows, two key groups): half the L2 -> LDS traffic per row, one barrier per tile,
//     K two tiles and V one tile ahead, as in the general kernel.
// All query heads of a KV head are packed into a workgroup's rows whatever the caller's pack, so
// K/V is read once per group of heads, also for group sizes that do not divide block_m. A row's
// arithmetic depends on BN, KG and the split only, so packed and unpacked calls stay equal bit for
// bit. VARIANT is 0, or kVariantMaskEveryTile in the measurement library.
#pragma once

#include "attn_fwd_common.hpp"
#include "attn_fwd_schedule.hpp"

namespace fa2 {

// s_waitcnt as a fence: no memory access moves across it.
template <int N>
__device__ __forceinline__ void wait_vm_fence() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int DT, int D, int GW, int BN, bool CAUSAL, int VARIANT = 0>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2)))
void attn_wave_split_kernel(const Params p) {
  using E = Elem<DT>;
  constexpr bool kMaskEveryTile = (VARIANT & kVariantMaskEveryTile) != 0;
  constexpr int KG = 4 / GW;         // key groups
  constexpr int BUFS = GW == 1 ? 1 : 2;  // K (and V) tiles in LDS per group
  constexpr int KS = D / 16;         // 16-dim k-steps of S^T = K Q^T
  constexpr int DB = (D + 31) / 32;  // 32-dim row blocks of O^T
  constexpr int NB = BN / 32;        // 32-key row blocks of S^T
  constexpr int NT = BN / 16;        // 16-key k-steps of O^T
  constexpr int CPR = D / 8;         // 16-byte chunks per K / V row
  constexpr int TCH = BN * CPR;      // chunks per K (or V) tile
  constexpr int NI = TCH / 64;       // load instructions per tile
  constexpr int JW = NI / GW;        // ... per wave
  static_assert(TCH % (64 * GW) == 0, "a tile must be whole 1 KiB load instructions of every wave");
  constexpr int QPR = D / 4;         // 16-byte pieces of an fp32 output row

  // K/V buffers; after the loop, the groups' O (fp32 rows, 16-byte pieces XOR-swizzled by row)
  constexpr int kKvChunks = KG * BUFS * 2 * TCH;
  constexpr int kMergeChunks = KG * GW * 32 * QPR;
  __shared__ u32x4 lds[kKvChunks > kMergeChunks ? kKvChunks : kMergeChunks];
  __shared__ float sm[KG][GW * 32][3];  // m, l, exact l of every group's rows

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 31;
  const int g = lane >> 5;
  const int grp = wave / GW, gwave = wave % GW;

  const int rows = p.n_q * p.group;  // row r: position r / group, head r % group of the KV head
  const SplitProgram pr = split_program<CAUSAL>(p, (int)blockIdx.x);
  const int split = pr.split, b = pr.b, hkv = pr.hkv;
  const int row0 = pr.tile * (32 * GW);  // this workgroup's rows [row0, row_end)
  const int row_end = min(row0 + 32 * GW, rows);

  // ---- this lane's row; rows past the last repeat it and are never stored
  const int r = min(row0 + gwave * 32 + c, rows - 1);
  const int pos = r / p.group;
  u32x4 qreg[KS];
  {
    const int head = hkv * p.group + (r - pos * p.group);
    const uint16_t* qrow = p.q + b * p.sqb + head * p.sqh + (int64_t)pos * p.sqn + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qreg[ks] = *(const u32x4*)(qrow + 16 * ks);
  }
  // the last key the row sees, and the end of the keys that every row of the workgroup sees
  const int last_key = CAUSAL ? min(pos, p.n_kv - 1) : p.n_kv - 1;
  const int full_end = CAUSAL ? min(row0 / p.group + 1, p.n_kv) : p.n_kv;

  // ---- this group's tiles: grp, grp + KG, ... of the split's [t_begin, t_begin + n_tiles)
  const int kv_end = CAUSAL ? min((row_end - 1) / p.group + 1, p.n_kv) : p.n_kv;
  const int all_tiles = (kv_end + BN - 1) / BN;
  const int t_begin = split * p.split_tiles;
  const int n_tiles = p.splits > 1 ? min(p.split_tiles, all_tiles - t_begin) : all_tiles;
  const int count = (n_tiles - grp + KG - 1) / KG;
  auto key_of = [&](int i) { return (t_begin + grp + i * KG) * BN; };  // first key of tile i

  const char* kbase = (const char*)(p.k + b * p.skb + hkv * p.skh);
  const char* vbase = (const char*)(p.v + b * p.svb + hkv * p.svh);
  uint32_t koff[JW], voff[JW];
#pragma unroll
  for (int j = 0; j < JW; ++j) {
    const int P = (gwave * JW + j) * 64 + lane;
    const int row = P / CPR, col = P % CPR;
    koff[j] = (uint32_t)(row * p.skn + (col ^ k_key<D>(pi_row(row & 31) & 15)) * 8) * 2u;
    voff[j] = (uint32_t)(row * p.svn + (col ^ v_key<D>(row & 15)) * 8) * 2u;
  }
  // The resource of the group's tile i covers that tile's rows only, at most to the last key (the
  // host bounds the row stride so that this stays below 2^31 bytes). Past the group's last tile it
  // covers nothing: the loads write zeros to LDS and read no memory, so a tile is always JW loads
  // and the counted waits below stay exact.
  auto rsrc_at = [&](const char* base, int64_t stride, int i) {
    const int n0 = i < count ? key_of(i) : 0;
    const uint32_t stride2 = (uint32_t)stride * 2u;
    const uint32_t nrows = (uint32_t)min(p.n_kv - n0, BN);  // 1 .. BN
    const uint32_t bytes = i < count ? (nrows - 1u) * stride2 + (uint32_t)D * 2u : 0u;
    return make_desc(base + (uint64_t)(uint32_t)n0 * stride2, bytes);
  };
  const FA2_LDS char* gbuf = (const FA2_LDS char*)(lds + grp * BUFS * 2 * TCH);
  auto kbuf = [&](int i) { return gbuf + (BUFS == 1 ? 0 : (i & 1) * TCH * 16); };
  auto vbuf = [&](int i) { return kbuf(i) + BUFS * TCH * 16; };
  auto issue_k = [&](int i) {
    const auto rs = rsrc_at(kbase, p.skn, i);
#pragma unroll
    for (int j = 0; j < JW; ++j) load_lds16(rs, koff[j], lds_addr(kbuf(i) + (gwave * JW + j) * 1024));
  };
  auto issue_v = [&](int i) {
    const auto rs = rsrc_at(vbase, p.svn, i);
#pragma unroll
    for (int j = 0; j < JW; ++j) load_lds16(rs, voff[j], lds_addr(vbuf(i) + (gwave * JW + j) * 1024));
  };

  // ---- LDS operand reads, as in attn_fwd_kernel.hpp
  const int kk = k_key<D>(c & 15);
  const int vj = (lane & 15) >> 2;
  const int vq = lane & 3;
  const int vsig = ((vq & 1) << 1) | ((vq & 2) >> 1);
  const int vdh = (D == 16) ? 0 : ((lane >> 4) & 1);
  uint32_t koffs[KS], voffs[2][DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koffs[ks] = (uint32_t)((pi_row(c) * CPR + ((2 * ks + g) ^ kk)) * 16);
#pragma unroll
  for (int rr = 0; rr < 2; ++rr)
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int row = 8 * g + 4 * rr + vj;
      const int chunk = (4 * db + 2 * vdh + (vsig >> 1)) ^ v_key<D>(row);
      voffs[rr][db] = (uint32_t)(row * (D * 2) + chunk * 16 + (vsig & 1) * 8);
    }
  auto k_operand = [&](int i, int ks, int nb) {
    return *(const u32x4 FA2_LDS*)(kbuf(i) + koffs[ks] + nb * 32 * CPR * 16);
  };
  auto v_operand = [&](int i, int t, int db) {
    const u32x2 lo = lds_read_tr(vbuf(i) + voffs[0][db] + t * 16 * D * 2);
    const u32x2 hi = lds_read_tr(vbuf(i) + voffs[1][db] + t * 16 * D * 2);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };

  // ---- the online softmax of one tile, base 2, with a lazily moved reference (fa2/kernel.py:81-98);
  // P is rounded to the input type and l sums the rounded P (attn_fwd_kernel.hpp says why)
  float m_i = -INFINITY, l_i = 0.f, l_exact = 0.f;
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x16{};
  const float qk_scale = p.qk_scale;
  const bool want_exact = p.lse != nullptr;
  auto softmax = [&](f32x16 (&s)[NB], u32x4 (&pb)[NT], int n0) {
    if (kMaskEveryTile || n0 + BN > full_end) {
      const int lim = last_key - n0 - 8 * g;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int x = 0; x < 16; ++x)
          if (nb * 32 + 16 * (x / 8) + (x % 8) > lim) s[nb][x] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int x = 0; x < 16; ++x) mx = fmaxf(mx, s[nb][x]);
    mx = pair_max(mx) * qk_scale;
    const bool grow = mx > m_i + kRescaleTau;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float m_new = grow ? mx : m_i;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m_i - m_new) : 1.0f;
      l_i *= alpha;
      l_exact *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) acc[db] *= alpha;
      m_i = m_new;
    }
    // a row that has seen no key in this group's tiles yet (reference -inf) gets weights 0, not NaN
    const float m_ref = m_i == -INFINITY ? 0.f : m_i;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int x = 0; x < 16; ++x)
        s[nb][x] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[nb][x], qk_scale, -m_ref));
    if (want_exact) l_exact += lane_sum(s);
    float rs0 = 0.f, rs1 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int nb = t >> 1, h = t & 1;
      pb[t] = u32x4{E::pack2(s[nb][8 * h + 0], s[nb][8 * h + 1]),
                    E::pack2(s[nb][8 * h + 2], s[nb][8 * h + 3]),
                    E::pack2(s[nb][8 * h + 4], s[nb][8 * h + 5]),
                    E::pack2(s[nb][8 * h + 6], s[nb][8 * h + 7])};
      rs0 = E::sum2(pb[t][0], rs0);
      rs1 = E::sum2(pb[t][1], rs1);
      rs0 = E::sum2(pb[t][2], rs0);
      rs1 = E::sum2(pb[t][3], rs1);
    }
    l_i += rs0 + rs1;
  };

  if constexpr (GW == 1) {
    issue_k(0);
    issue_v(0);
    // Q is waited for here, before the loop: the compiler does not count the asm loads above, so
    // its own wait for Q is for everything in flight, and inside the loop it would come every time
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qreg[ks]));
    for (int i = 0; i < count; ++i) {
      // S^T = K Q^T (fa2/kernel.py:75-79)
      wait_vm_fence<NI>();  // K_i has landed; V_i may be in flight
      u32x4 kop[KS][NB];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) kop[ks][nb] = k_operand(i, ks, nb);
      wait_lds_fence();  // the operands have left the buffer: refill it
      issue_k(i + 1);
      f32x16 s[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) s[nb] = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s[nb] = E::mma(kop[ks][nb], qreg[ks], s[nb]);
      u32x4 pb[NT];
      softmax(s, pb, key_of(i));
      // O^T += V^T P^T (fa2/kernel.py:100-105)
      wait_vm_fence<NI>();  // V_i has landed; K_{i+1} may be in flight
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = E::mma(v_operand(i, t, db), pb[t], acc[db]);
      wait_lds_fence();
      issue_v(i + 1);
    }
  } else {
    // One barrier per tile, between the two products, as in attn_fwd_kernel.hpp's loop; the groups
    // run the same number of trips (a group with fewer tiles idles through the last).
    constexpr int LA_S = KS < 4 ? KS : 4;  // k-steps of K operands read ahead
    constexpr int NPV = NT * DB;           // MFMAs of the PV product
    constexpr int LA_V = NPV < 4 ? NPV : 4;
    constexpr int NKP = LA_S * NB;         // K operand reads prefetched during PV
    const int n_iter = (n_tiles + KG - 1) / KG;
    // tiles that start past every row of the wave add exact zeros: their products are skipped
    const int wave_last = __builtin_amdgcn_readlane(last_key, 31);  // rows grow with the lane
    const int first = key_of(0);
    const int n_active = wave_last < first ? 0 : min(count, (wave_last - first) / (KG * BN) + 1);
    issue_k(0);
    issue_v(0);
    issue_k(1);
    wait_vm_fence<2 * JW>();
    __syncthreads();
    u32x4 kop[LA_S][NB];
#pragma unroll
    for (int ks = 0; ks < LA_S; ++ks)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        kop[ks][nb] = *(const volatile u32x4 FA2_LDS*)(kbuf(0) + koffs[ks] + nb * 32 * CPR * 16);
    for (int j = 0; j < n_active; ++j) {
      __builtin_amdgcn_s_setprio(1);
      f32x16 s[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) s[nb] = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int slot = ks % LA_S;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s[nb] = E::mma(kop[slot][nb], qreg[ks], s[nb]);
        if (ks + LA_S < KS) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) kop[slot][nb] = k_operand(j, ks + LA_S, nb);
        }
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        __builtin_amdgcn_sched_group_barrier(0x008, NB, 0);
        if (ks + LA_S < KS) __builtin_amdgcn_sched_group_barrier(0x100, NB, 0);
      }
      __builtin_amdgcn_s_setprio(0);
      wait_vm_fence<0>();  // this wave's loads of V_j and K_{j+1} have landed
      __syncthreads();     // ... every wave's; and every wave is done with K_j
      if (j + 2 < count) issue_k(j + 2);
      if (j + 1 < count) issue_v(j + 1);
      u32x4 va[LA_V], pb[NT];
#pragma unroll
      for (int x = 0; x < LA_V; ++x) va[x] = v_operand(j, x / DB, x % DB);
      softmax(s, pb, key_of(j));
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int x = 0; x < NPV; ++x) {
        acc[x % DB] = E::mma(va[x % LA_V], pb[x / DB], acc[x % DB]);
        if (x + LA_V < NPV) va[x % LA_V] = v_operand(j, (x + LA_V) / DB, (x + LA_V) % DB);
        // K_{j+1}'s first operands (a harmless stale read after the last tile)
#pragma unroll
        for (int y = x * NKP / NPV; y < (x + 1) * NKP / NPV; ++y)
          kop[y / NB][y % NB] = k_operand(j + 1, y / NB, y % NB);
      }
#pragma unroll
      for (int x = 0; x < NPV; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        const int nreads = (x + LA_V < NPV ? 2 : 0) + ((x + 1) * NKP / NPV - x * NKP / NPV);
#pragma unroll
        for (int y = 0; y < nreads; ++y) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    for (int j = n_active; j < n_iter; ++j) {
      wait_vm_fence<0>();
      __syncthreads();
      if (j + 2 < count) issue_k(j + 2);
      if (j + 1 < count) issue_v(j + 1);
    }
  }

  // ---- merge the groups through LDS: O^T blocks as 16-byte pieces [group][row][4 dims], then
  // every thread folds the groups of its pieces
  wait_vm_fence<0>();
  __syncthreads();  // every wave is done with every K/V buffer
  FA2_LDS f32x4* ob = (FA2_LDS f32x4*)lds;
  auto piece = [&](int group, int row, int q) {
    return (group * GW * 32 + row) * QPR + (q ^ (row & (QPR < 8 ? QPR - 1 : 7)));
  };
  {
    const int wr = gwave * 32 + c;  // the row inside the workgroup
    const float l = pair_sum(l_i);
    const float lx = want_exact ? pair_sum(l_exact) : l;
    if (row0 + wr < row_end) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int q = 8 * db + 4 * (h >> 1) + 2 * g + (h & 1);  // dims 4 q .. 4 q + 3
          if (q < QPR) {
            f32x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = acc[db][4 * h + e];
            ob[piece(grp, wr, q)] = x;
          }
        }
      if (g == 0) {
        sm[grp][wr][0] = m_i;
        sm[grp][wr][1] = l;
        sm[grp][wr][2] = lx;
      }
    }
  }
  __syncthreads();
  for (int t = tid; t < (row_end - row0) * QPR; t += 256) {
    const int wr = t / QPR, q = t % QPR;
    float m = -INFINITY, l = 0.f, lx = 0.f;
#pragma unroll
    for (int x = 0; x < KG; ++x) m = fmaxf(m, sm[x][wr][0]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < KG; ++x) {
      const float mw = sm[x][wr][0];
      const float w = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - m);
      l = __builtin_fmaf(w, sm[x][wr][1], l);
      lx = __builtin_fmaf(w, sm[x][wr][2], lx);
      const f32x4 v = ob[piece(x, wr, q)];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(w, v[e], o[e]);
    }
    const float inv_l = 1.0f / l;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] *= inv_l;
    const int opos = (row0 + wr) / p.group;
    const int head = hkv * p.group + (row0 + wr - opos * p.group);
    const int64_t row_index = ((int64_t)b * p.h_q + head) * p.n_q + opos;  // in [B, H_q, N_q]
    if (p.splits > 1) {  // split-KV partials for attn_fwd_combine.hip
      *(f32x4*)(p.part_o + ((int64_t)split * p.part_rows + row_index) * D + 4 * q) = o;
      if (q == 0) {
        p.part_lse[(int64_t)split * p.part_rows + row_index] = m + log2f(l);
        if (p.lse) p.part_lse_exact[(int64_t)split * p.part_rows + row_index] = m + log2f(lx);
      }
    } else {
      uint16_t* orow = p.o + b * p.sob + head * p.soh + (int64_t)opos * p.son + 4 * q;
      *(u32x2*)orow = u32x2{E::pack2(o[0], o[1]), E::pack2(o[2], o[3])};
      if (p.lse && q == 0) p.lse[row_index] = (m + log2f(lx)) * kLn2;
    }
  }
}

}  // namespace fa2
