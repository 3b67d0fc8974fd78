// The body of fa_fwd16_kernel (flash_attn_fwd.hip: dense attention at head_dim 128 on the 16x16x32 matrix instruction)
// in two other shapes of work.  NW waves of 32 rows each walk key tiles of BN keys.
//
// KS 1: a workgroup that keeps its CU and goes from one tile of rows to the next (fa16_loop_kernel states why).
//
// KS > 1: workgroups that own fewer query rows: the waves form KS groups that share the same NW / KS * 32 query rows, each
// taking BN / KS keys of every tile with a running softmax of its own; the groups' sums and outputs are added up in LDS
// at the end, in 32 bits.  Why: the launch time of fa_fwd16_kernel is rounds of 256 workgroups of 256 rows, and a round
// that is a quarter full takes as long as a full one.  A workgroup of 128 (KS 2) or 64 rows (KS 4) has half or a quarter
// of the matrix and vector work per tile for the same number of waves: its walk over the keys takes 0.62 or 0.46 of the
// time (KS 4: 1.3 us per 128 keys, the L2 -> LDS stream of 64 KiB at 50 GB/s per CU; whole tiles: 3.0 us, matrix and
// vector issue).  No workspace, no second launch.
//
// KEYMASK: a boolean mask row shared by all queries of a (batch, head), as GEN 3 of fa_fwd16_kernel.
#pragma once
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "fa_params.hpp"

namespace msd {

// LDS of a workgroup: the tile stages; the groups' hand-over and the output staging reuse them (KS 1: staging of its own)
template <int D, int KS>
constexpr int fa16_flex_lds(int nw, int bn) {
  const int stages = 4 * bn * 2 * D, part = nw * ((D / 16 - D / 16 / KS) * 2048 + 1024) + nw * 32 * (2 * D / KS + 8);
  return KS == 1 ? stages + nw * 4096 : stages > part ? stages : part;
}

#if defined(__HIP_DEVICE_COMPILE__)
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>)
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// item: the first tile of NW / KS * 32 query rows, numbered through the heads ((batch, head) * row_tiles + tile; rows at
// or beyond p.Sq do not exist); part: KS > 1, which part of a tile of NW * 32 rows it is.  KS 1: the workgroup goes on with
// the tiles item + 32, item + 64, ... below `end`.
// LDS: K stages at 0 and BN * 256 bytes, V stages behind them, with KS 1 the output staging behind those; swizzles and
// operand layouts as in fa_fwd16_kernel.
//
// D: head_dim, 128 or 64 (fa_fwd16_d64_kernel's layouts: rows of 128 bytes, K chunk p of row r at p ^ ((r >> 1) & 7), V
// chunk p at p ^ ((r >> 1) & 3)).
template <int DT, int NW, int BN, int KS, bool KEYMASK, int D = 128>
__device__ __forceinline__ void fa16_flex_body(const FaParams& p, MSD_LDS char* smem, int item, int part, int end) {
  using E = Elem<DT>;
  using T = typename E::type;
  using X8 = typename E::x8;
  static_assert(D == 128 || (D == 64 && KS > 1), "head_dim");
  constexpr int kRowBytes = 2 * D, kDmaRows = 1024 / kRowBytes, NDB = D / 16, NKS = D / 32, kTileBytes = BN * kRowBytes;
  constexpr int RG = NW / KS;         // waves side by side over the query rows
  constexpr int kKeys = BN / KS;      // keys of a tile that one wave takes
  constexpr int NKB = kKeys / 16;     // its 16-key blocks
  constexpr int NJ = kKeys / 32;      // its 32-key steps of the second product
  static_assert(NKB % 2 == 0 && NW % KS == 0 && (4 * NW) % 16 == 0, "whole operand groups");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int rg = wave % RG, kg_i = wave / RG;
  constexpr bool LOOP = KS == 1;
  const int Sq = p.Sq, Skv = p.Skv;
  const int row_tiles = (Sq + NW * 32 - 1) / (NW * 32);
  // the tile at hand, and with LOOP the one after it
  int b, n, row0, b_nx = 0, n_nx = 0, row0_nx = 0;
  auto locate = [&](int it, int& ib, int& in, int& irow) __attribute__((always_inline)) {
    const int bn = it / row_tiles;
    ib = bn / p.N;
    in = bn - ib * p.N;
    irow = (it - bn * row_tiles) * (NW * 32) + part * (NW / KS * 32) + rg * 32;
  };
  locate(item, b, n, row0);

  // ---- staging (LDS-DMA) -------------------------------------------------------------------------------------
  const int group = p.N / p.Nkv;
  const int k_range = (int)(((long long)(Skv - 1) * p.k_ss + D) * 2), v_range = (int)(((long long)(Skv - 1) * p.v_ss + D) * 2);
  auto k_base = [&](int ib, int in) __attribute__((always_inline)) { return (const T*)p.k + ib * p.k_sb + (in / group) * p.k_sn; };
  auto v_base = [&](int ib, int in) __attribute__((always_inline)) { return (const T*)p.v + ib * p.v_sb + (in / group) * p.v_sn; };
  const T *kg = k_base(b, n), *vg = v_base(b, n), *kg_nx = kg, *vg_nx = vg;
  const int k_row_bytes = (int)p.k_ss * 2, v_row_bytes = (int)p.v_ss * 2;
  int k_voff, v_voff;
  {
    const int row = kDmaRows * wave + lane / (kRowBytes / 16);  // groups of one wave lie kDmaRows * NW rows apart: same swizzles
    const int pc = lane % (kRowBytes / 16);
    const int ksw = D == 128 ? row & 15 : (row >> 1) & 7, vsw = D == 128 ? row & 7 : (row >> 1) & 3;
    k_voff = row * k_row_bytes + ((pc ^ ksw) << 4);
    v_voff = row * v_row_bytes + (((((pc >> 1) ^ vsw) << 1) | (pc & 1)) << 4);
  }
  auto load_tile = [&](const T* kp, const T* vp, int key0, int stage) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, k_range, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, v_range, 0x00020000);
#pragma unroll
    for (int i = 0; i < BN / kDmaRows / NW; ++i) {
      const int grp = i * NW + wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rsrc, (MSD_LDS void*)(smem + stage * kTileBytes + grp * 1024), 16, k_voff,
                                               (key0 + i * kDmaRows * NW) * k_row_bytes, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rsrc, (MSD_LDS void*)(smem + (2 + stage) * kTileBytes + grp * 1024), 16,
                                               v_voff, (key0 + i * kDmaRows * NW) * v_row_bytes, 0, 0);
    }
  };

  // ---- Q^T operand, resident: requested here, converted at the start of its tile ------------------------------------
  X8 qf[2][NKS];
  auto load_q = [&](int ib, int in, int irow) __attribute__((always_inline)) {
    const T* qg = (const T*)p.q + ib * p.q_sb + in * p.q_sn;
    int c = lane & 15, g = lane >> 4;
    if constexpr (LOOP) asm volatile("" : "+v"(c), "+v"(g));  // (recomputed for every tile, not kept in registers)
#pragma unroll
    for (int nq = 0; nq < 2; ++nq) {
      const int qrow = irow + nq * 16 + c;
      const T* src = qg + (long long)(qrow < Sq ? qrow : 0) * p.q_ss + 8 * g;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) qf[nq][ks] = *(const X8*)(src + 32 * ks);
    }
  };
  f32x4_t oacc[NDB][2], negm[2], lt[2];
  float l_run[2];
  X8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = E::from_float(1.f);

  // per-lane parts of the LDS read addresses (the wave's keys start at row kg_i * kKeys, a multiple of 16)
  unsigned k_lds[NKS], v_lds[4];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    k_lds[ks] = (unsigned)(uintptr_t)smem + (kg_i * kKeys + c) * kRowBytes + (((4 * ks + g) ^ (D == 128 ? c : c >> 1)) << 4);
#pragma unroll
  for (int db = 0; db < 4; ++db)
    v_lds[db] = (unsigned)(uintptr_t)smem + 2 * kTileBytes + (kg_i * kKeys + 4 * g + (c >> 2)) * kRowBytes +
                ((db ^ (D == 128 ? 4 * (g & 1) + (c >> 2) : ((4 * g + (c >> 2)) >> 1) & 3)) << 5) + 8 * (c & 3);

  const int tiles = (Skv + BN - 1) / BN;
  load_q(b, n, row0);
  load_tile(kg, vg, 0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  bool first = true;

  // ---- key mask: words of visible keys of the current tile, bit l of word j = key 4 * l + j -----------------------------
  unsigned kvis[4] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu}, kraw = 0;
  const unsigned char* mask_g = nullptr;
  auto mask_request = [&](int key0) __attribute__((always_inline)) {
    if constexpr (KEYMASK) {
      kraw = 0;
      const int k4 = key0 + 4 * (lane & (BN / 4 - 1));
      if (key0 + BN <= Skv) {
        __builtin_memcpy(&kraw, mask_g + k4, 4);  // (any alignment)
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned byte = mask_g[min(k4 + j, Skv - 1)];
          kraw |= (k4 + j < Skv ? byte : 0u) << (8 * j);
        }
      }
    }
  };
  auto mask_reduce = [&]() __attribute__((always_inline)) {
    if constexpr (KEYMASK) {
#pragma unroll
      for (int j = 0; j < 4; ++j)  // the wave's own keys, from bit 0 on
        kvis[j] = (unsigned)__builtin_amdgcn_ballot_w64(lane < BN / 4 && ((kraw >> (8 * j)) & 0xffu) != 0) >> (kg_i * (kKeys / 4));
    }
  };
  constexpr unsigned kOwn = (unsigned)((1ull << (kKeys / 4)) - 1);

  // next_tile: the first key of the tile to request, of the workgroup's next tile of rows with `other`; < 0: none
  auto tile_step = [&](auto stage_c, const int key0, const int next_tile, const bool other) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_c)::value;
    if (next_tile >= 0) load_tile(other ? kg_nx : kg, other ? vg_nx : vg, next_tile, stage ^ 1);
    const int next_key0 = other ? -1 : next_tile;
    const unsigned kv_all = kvis[0] & kvis[1] & kvis[2] & kvis[3] & kOwn;
    const int key_w = key0 + kg_i * kKeys;  // the wave's first key

    // S^T = K Q^T: operand groups of 2 key blocks of one 32-wide head_dim step, kAhead groups ahead of their use
    f32x4_t sacc[NKB][2];
    constexpr int kPer = NKB / 2, kGroups = NKS * kPer, kAhead = kGroups > 3 ? 3 : kGroups - 1;
    X8 afrag[kAhead + 1][2];
    auto k_read = [&](auto gi_c, X8(&dst)[2]) __attribute__((always_inline)) {
      constexpr int gi = decltype(gi_c)::value, ks = gi / kPer, qu = gi % kPer;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        dst[i] = *(MSD_LDS const X8*)(uintptr_t)(k_lds[ks] + stage * kTileBytes + (2 * qu + i) * 16 * kRowBytes);
    };
    static_for<kAhead>([&](auto gi_c) __attribute__((always_inline)) { k_read(gi_c, afrag[decltype(gi_c)::value]); });
    static_for<kGroups>([&](auto gi_c) __attribute__((always_inline)) {
      constexpr int gi = decltype(gi_c)::value, ks = gi / kPer, qu = gi % kPer;
      if constexpr (gi + kAhead < kGroups)
        k_read(std::integral_constant<int, gi + kAhead>{}, afrag[(gi + kAhead) % (kAhead + 1)]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int nq = 0; nq < 2; ++nq)
          sacc[2 * qu + i][nq] =
              E::mfma16(afrag[gi % (kAhead + 1)][i], qf[nq][ks], ks == 0 ? negm[nq] : sacc[2 * qu + i][nq]);
    });
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int gi = 0; gi < kGroups - kAhead; ++gi) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);

    if (key_w + kKeys > Skv) {  // keys past the end of the sequence (last tile only)
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (key_w + 16 * kb + 4 * g + i >= Skv) {
            sacc[kb][0][i] = -INFINITY;
            sacc[kb][1][i] = -INFINITY;
          }
    }
    if constexpr (KEYMASK) {
      if (kv_all != kOwn) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned w = kvis[i] >> g;  // key 16 * kb + 4 * g + i is bit 4 * kb + g of word i
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
            if (!((w >> (4 * kb)) & 1u)) {
              sacc[kb][0][i] = -INFINITY;
              sacc[kb][1][i] = -INFINITY;
            }
        }
      }
    }

    // online softmax (exp2 domain, lazily moved reference maximum; see fa_fwd_kernel)
    X8 pf[2][NJ];
    bool seen = !KEYMASK;
#pragma unroll
    for (int nq = 0; nq < 2; ++nq) {
      float mx = sacc[0][nq][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[kb][nq][i]);
      if constexpr (KEYMASK) seen = seen || __builtin_amdgcn_ballot_w64(mx > -INFINITY) != 0;
      l_run[nq] += lt[nq][0];
      if constexpr (NKB == 8) {  // (see cond_rescale_fa16)
        float delta = 0.f, alpha = 1.f;
        int moved = 0;
        if (first || __builtin_amdgcn_ballot_w64(mx > kTau) != 0) {
          mx = quarter_max(mx);
          delta = first ? mx : fmaxf(mx, 0.f);
          delta = (delta == -INFINITY) ? 0.f : delta;
          alpha = first ? 1.f : fast_exp2(-delta);
          moved = 1;
        }
        cond_rescale_fa16(__builtin_amdgcn_readfirstlane(moved), delta, alpha, l_run[nq], negm[nq], sacc[0][nq], sacc[1][nq],
                          sacc[2][nq], sacc[3][nq], sacc[NKB - 4][nq], sacc[NKB - 3][nq], sacc[NKB - 2][nq],
                          sacc[NKB - 1][nq], oacc[0][nq], oacc[1][nq], oacc[2][nq], oacc[3][nq], oacc[4][nq], oacc[5][nq],
                          oacc[6][nq], oacc[7][nq]);
      } else if (first || __builtin_amdgcn_ballot_w64(mx > kTau) != 0) {
        mx = quarter_max(mx);
        float delta = first ? mx : fmaxf(mx, 0.f);
        delta = (delta == -INFINITY) ? 0.f : delta;
        // (first tile: sums and outputs are still zero; 2^-delta would overflow for rows far below zero and 0 * inf is NaN)
        const float alpha = first ? 1.f : fast_exp2(-delta);
        l_run[nq] *= alpha;
#pragma unroll
        for (int i = 0; i < 4; ++i) negm[nq][i] -= delta;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) sacc[kb][nq][i] -= delta;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[db][nq][i] *= alpha;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        X8 pk;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          pk[t] = E::from_float(fast_exp2(sacc[2 * j][nq][t]));
          pk[4 + t] = E::from_float(fast_exp2(sacc[2 * j + 1][nq][t]));
        }
        pf[nq][j] = pk;
      }
    }

    constexpr int NH = NDB / 4;  // steps per 32 keys
    // O^T += V^T P^T: steps of (32 keys) x (4 head_dim blocks), V^T fragments requested one step ahead
    s16x4_t vf[2][8];
    auto issue = [&](auto step_c, s16x4_t(&dst)[8]) __attribute__((always_inline)) {
      constexpr int s = decltype(step_c)::value, j = s / NH, dbh = s % NH;
      constexpr int off = stage * kTileBytes + 32 * j * kRowBytes;
#pragma unroll
      for (int d4 = 0; d4 < 4; ++d4) {
        const unsigned a = v_lds[d4] ^ (dbh << 7);
        dst[2 * d4] = lds_read_tr16_async<off>(a);
        dst[2 * d4 + 1] = lds_read_tr16_async<off + 16 * kRowBytes>(a);
      }
    };
    if constexpr (KEYMASK) {
      if (next_key0 >= 0) mask_request(next_key0);  // lands during the second product
    }
    issue(std::integral_constant<int, 0>{}, vf[0]);
    static_for<NH * NJ>([&](auto step_c) __attribute__((always_inline)) {
      constexpr int s = decltype(step_c)::value, j = s / NH, dbh = s % NH;
      if constexpr (s + 1 < NH * NJ) {
        issue(std::integral_constant<int, s + 1>{}, vf[(s + 1) & 1]);
        lds_wait_tr<8>(vf[s & 1]);
      } else {
        lds_wait_tr<0>(vf[s & 1]);
      }
#pragma unroll
      for (int d4 = 0; d4 < 4; ++d4) {
        union { s16x4_t s2[2]; X8 x; } u;
        u.s2[0] = vf[s & 1][2 * d4];
        u.s2[1] = vf[s & 1][2 * d4 + 1];
#pragma unroll
        for (int nq = 0; nq < 2; ++nq) oacc[4 * dbh + d4][nq] = E::mfma16(u.x, pf[nq][j], oacc[4 * dbh + d4][nq]);
      }
      if constexpr (dbh == 0) {
#pragma unroll
        for (int nq = 0; nq < 2; ++nq)
          lt[nq] = E::mfma16(ones, pf[nq][j], j == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : lt[nq]);
      }
    });
    first = first && !seen;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the next tile has landed
    mask_reduce();
    __syncthreads();
  };
  for (;;) {
  if constexpr (KEYMASK) {
    mask_g = p.mask + b * p.m_sb + n * p.m_sn;
    mask_request(0);
    mask_reduce();
  }
#pragma unroll
  for (int nq = 0; nq < 2; ++nq) {
    int cc = c;
    if constexpr (LOOP) asm volatile("" : "+v"(cc));
    const bool ok = row0 + nq * 16 + cc < Sq;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      X8 v = qf[nq][ks];
      if (!ok) v = X8{0};
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = E::from_float((float)v[j] * p.scale_log2);
      qf[nq][ks] = v;
    }
    l_run[nq] = 0.f;
    negm[nq] = lt[nq] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int db = 0; db < NDB; ++db) oacc[db][nq] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  first = true;
  bool more = false;
  unsigned touched = 0;
  if constexpr (LOOP) {
    more = item + 32 < end;
    if (more) {
      locate(item + 32, b_nx, n_nx, row0_nx);
      kg_nx = k_base(b_nx, n_nx);
      vg_nx = v_base(b_nx, n_nx);
      // a word of every 128-byte line of the next rows of q, so that they wait in the L2
      const int qrow = min(row0_nx - rg * 32 + (tid >> 1), Sq - 1);
      touched = *(const unsigned*)((const T*)p.q + b_nx * p.q_sb + n_nx * p.q_sn + (long long)qrow * p.q_ss + (tid & 1) * 64);
    }
  }
  for (int t = 0; t < tiles; t += 2) {
    tile_step(std::integral_constant<int, 0>{}, t * BN, t + 1 < tiles ? (t + 1) * BN : -1, false);
    // (an even number of key tiles: the last step requests the first key tile of the next rows)
    if (t + 1 < tiles)
      tile_step(std::integral_constant<int, 1>{}, (t + 1) * BN, t + 2 < tiles ? (t + 2) * BN : (LOOP && more ? 0 : -1),
                LOOP && t + 2 >= tiles);
  }
  if constexpr (LOOP) {
    asm volatile("" ::"v"(touched));
    if (more) {  // (an odd number: it goes into the stage of the last step, which no wave reads any more)
      load_q(b_nx, n_nx, row0_nx);
      if (tiles & 1) load_tile(kg_nx, vg_nx, 0, 0);
    }
  }

  // ---- the groups' partial results (KS > 1) --------------------------------------------------------------------------
  // Every wave ends up with all 32 rows of its row group and NDB / KS of the output's 16-wide blocks: it hands the other
  // blocks to the waves that own them (16 bytes per lane and block, the accumulator layout as it is) together with its
  // reference maxima and sums.  A group that saw no key has sum 0 and no say in the maximum.
  constexpr int DB = NDB / KS;                       // output blocks a wave stores
  constexpr int kPart = (NDB - DB) * 2 * 1024;       // bytes a wave hands out
  constexpr int kStat = KS > 1 ? 4 * 256 : 0;      // m and l of two column blocks, a dword per lane
  constexpr int kORow = 2 * 16 * DB + 8;           // a row of the output staging, padded
  constexpr int kOBase = KS > 1 ? NW * (kPart + kStat) : 0;
  static_assert(KS == 1 || kOBase + NW * 32 * kORow <= fa16_flex_lds<D, KS>(NW, BN), "fits");
  float l_tot[2], m_tot[2];
#pragma unroll
  for (int nq = 0; nq < 2; ++nq) {
    l_tot[nq] = l_run[nq] + lt[nq][0];
    m_tot[nq] = -negm[nq][0];
  }
  if constexpr (KS > 1) {
    MSD_LDS char* mine = smem + wave * (kPart + kStat);
    // block db belongs to group db / DB; slot of a block that is not the writer's: the blocks in order, its own left out
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const int owner = db / DB;
      const int slot = owner < kg_i ? db : db - DB;
      if (owner != kg_i) {
#pragma unroll
        for (int nq = 0; nq < 2; ++nq) *(MSD_LDS f32x4_t*)(mine + (slot * 2 + nq) * 1024 + lane * 16) = oacc[db][nq];
      }
    }
#pragma unroll
    for (int nq = 0; nq < 2; ++nq) {
      *(MSD_LDS float*)(mine + kPart + (2 * nq) * 256 + lane * 4) = m_tot[nq];
      *(MSD_LDS float*)(mine + kPart + (2 * nq + 1) * 256 + lane * 4) = l_tot[nq];
    }
    __syncthreads();
    f32x4_t own[DB][2];
#pragma unroll
    for (int k = 0; k < KS; ++k)
      if (k == kg_i) {
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int nq = 0; nq < 2; ++nq) own[d][nq] = oacc[k * DB + d][nq];
      }
#pragma unroll
    for (int nq = 0; nq < 2; ++nq) {
      float mk[KS], lk[KS], m = -INFINITY, l = 0.f;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        MSD_LDS const char* st = smem + (k * RG + rg) * (kPart + kStat) + kPart + (2 * nq) * 256 + lane * 4;
        mk[k] = *(MSD_LDS const float*)st;
        lk[k] = *(MSD_LDS const float*)(st + 256);
        if (lk[k] != 0.f) m = fmaxf(m, mk[k]);
      }
      f32x4_t sum[DB];
#pragma unroll
      for (int d = 0; d < DB; ++d) sum[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const float w = lk[k] != 0.f ? fast_exp2(mk[k] - m) : 0.f;
        l += w * lk[k];
        MSD_LDS const char* from = smem + (k * RG + rg) * (kPart + kStat);
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const int db = kg_i * DB + d;
          const int slot = kg_i < k ? db : db - DB;
          f32x4_t v = own[d][nq];
          if (k != kg_i) v = *(MSD_LDS const f32x4_t*)(from + (slot * 2 + nq) * 1024 + lane * 16);
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[d][i] += w * v[i];
        }
      }
#pragma unroll
      for (int d = 0; d < DB; ++d) oacc[d][nq] = sum[d];
      l_tot[nq] = l;
      m_tot[nq] = m;
    }
  }

  // ---- normalise, transpose the wave's rows through LDS, coalesced store ----------------------------------------------
  T* og = (T*)p.o + b * p.o_sb + n * p.o_sn;
  if constexpr (LOOP) {
    // 16 rows at a time through 4 KiB per wave behind the tile stages (which already fill with the next rows' keys):
    // 16-byte chunk k of row r sits at chunk k ^ r
    MSD_LDS char* ost = smem + 4 * BN * 256 + wave * 4096;
    int c = lane & 15, g = lane >> 4;
    asm volatile("" : "+v"(c), "+v"(g));
#pragma unroll
    for (int nq = 0; nq < 2; ++nq) {
      const float inv = l_tot[nq] > 0.f ? 1.f / l_tot[nq] : 0.f;
      const int qrow_l = row0 + nq * 16 + c;
      if (p.lse && g == 0 && qrow_l < Sq)
        p.lse[((long long)b * p.N + n) * Sq + qrow_l] =
            l_tot[nq] > 0.f ? m_tot[nq] * 0.6931471805599453f + __logf(l_tot[nq]) : -INFINITY;
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        typename E::x4 pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk[i] = E::from_float(oacc[db][nq][i] * inv);
        *(MSD_LDS typename E::x4*)(ost + c * 256 + (((2 * db + (g >> 1)) ^ c) << 4) + 8 * (g & 1)) = pk;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * i + g, qrow = row0 + nq * 16 + row;
        const i32x4_t v = *(MSD_LDS const i32x4_t*)(ost + row * 256 + ((c ^ row) << 4));
        if (qrow < Sq) *(i32x4_t*)(og + (long long)qrow * p.o_ss + c * 8) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (!more) return;
    item += 32;
    b = b_nx;
    n = n_nx;
    row0 = row0_nx;
    kg = kg_nx;
    vg = vg_nx;
    if (tiles & 1) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      __syncthreads();
    }
    continue;
  }
  MSD_LDS char* ost = smem + kOBase + wave * 32 * kORow;
#pragma unroll
  for (int nq = 0; nq < 2; ++nq) {
    const float inv = l_tot[nq] > 0.f ? 1.f / l_tot[nq] : 0.f;
    const int qrow_l = row0 + nq * 16 + c;
    if (p.lse && kg_i == 0 && g == 0 && qrow_l < Sq)
      p.lse[((long long)b * p.N + n) * Sq + qrow_l] =
          l_tot[nq] > 0.f ? m_tot[nq] * 0.6931471805599453f + __logf(l_tot[nq]) : -INFINITY;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      typename E::x4 pk;
#pragma unroll
      for (int i = 0; i < 4; ++i) pk[i] = E::from_float(oacc[d][nq][i] * inv);
      *(MSD_LDS typename E::x4*)(ost + (nq * 16 + c) * kORow + (16 * d + 4 * g) * 2) = pk;
    }
  }
  __builtin_amdgcn_wave_barrier();
  constexpr int kChunks = 2 * DB;  // 16-byte chunks of a row
#pragma unroll
  for (int i = 0; i < 32 * kChunks / 64; ++i) {
    const int ch = i * 64 + lane;
    const int row = ch / kChunks, c16 = ch % kChunks;
    const int qrow = row0 + row;
    const i32x2_t lo = *(MSD_LDS const i32x2_t*)(ost + row * kORow + c16 * 16);
    const i32x2_t hi = *(MSD_LDS const i32x2_t*)(ost + row * kORow + c16 * 16 + 8);
    if (qrow < Sq) *(i32x4_t*)(og + (long long)qrow * p.o_ss + kg_i * (16 * DB) + c16 * 8) = i32x4_t{lo[0], lo[1], hi[0], hi[1]};
  }
  return;
  }
}
#endif

}  // namespace msd
