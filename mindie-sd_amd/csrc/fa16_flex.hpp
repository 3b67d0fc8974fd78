// The body of fa_fwd16_kernel and fa_fwd16_d64_kernel (dense attention at head_dim 128 and 64 on the 16x16x32 matrix
// instruction) in two other shapes of work.  Eight waves walk key tiles of 128 keys as there, a wave owns NQ blocks of 16
// query rows.  The arithmetic of a block of 16 rows - the chains of matrix instructions, when its reference maximum moves,
// the rounding of its probabilities - is that of the kernels' whole tiles, so a row has the same bits in either.
//
// LOOP (NQ 2): a workgroup that keeps its CU and goes from one tile of 256 rows to the next (fa16_loop_kernel states why).
//
// Otherwise (NQ 1): a workgroup that owns part_rows (128 or 64) of a tile's 256 rows, 16 per wave; waves beyond them, or
// beyond the last row, only stage keys.  Why: the launch time of the kernels is rounds of 256 workgroups of 256 rows, and a
// round that is a quarter full takes as long as a full one.  What bounds it: every wave reads the whole key tile from LDS for
// its 16 rows, 512 KiB per 128 keys and half tile (1.75 us at 128 bytes a cycle; it takes 1.96, a whole tile 3.15 us of matrix
// and vector issue); a quarter tile takes 1.23 us, the L2 -> LDS stream of 64 KiB at 50 GB/s per CU.  (Head_dim 64: 1.15, 0.78 and
// 1.91 us.)  Groups of waves that split the keys of 32 rows read less and take 1.82 and 1.16 us, but add a row up in another order
// than the whole tiles of the same launch, so that equal problems of one batch came out with different bits.
//
// KEYMASK: a boolean mask row shared by all queries of a (batch, head), as GEN 3 of the kernels.
#pragma once
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "fa_params.hpp"

namespace msd {

// LDS of fa16_loop_kernel: the tile stages and the output staging behind them
constexpr int kFa16LoopLds = 4 * 128 * 256 + 8 * 16 * 256;

#if defined(__HIP_DEVICE_COMPILE__)
// The kernel's argument block (its only argument), to be read where it is needed: the compiler loads what it sees as one block
// up front and keeps it, and the bodies below then spill scalar registers into vector registers that their loops need.
typedef const __attribute__((address_space(4))) FaParams* FaArgs;
__device__ __forceinline__ FaArgs fa_args_here() {
  FaArgs a = (FaArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}

// the rescale of column block nq when its reference maximum moves (see cond_rescale_fa16)
template <int NQ>
__device__ __forceinline__ void fa16_rescale(int flag, float delta, float alpha, float& l, f32x4_t& negm, f32x4_t& s0, f32x4_t& s1,
                                             f32x4_t& s2, f32x4_t& s3, f32x4_t& s4, f32x4_t& s5, f32x4_t& s6, f32x4_t& s7,
                                             f32x4_t (&o)[8][NQ], int nq) {
  cond_rescale_fa16(flag, delta, alpha, l, negm, s0, s1, s2, s3, s4, s5, s6, s7, o[0][nq], o[1][nq], o[2][nq], o[3][nq], o[4][nq],
                    o[5][nq], o[6][nq], o[7][nq]);
}
template <int NQ>
__device__ __forceinline__ void fa16_rescale(int flag, float delta, float alpha, float& l, f32x4_t& negm, f32x4_t& s0, f32x4_t& s1,
                                             f32x4_t& s2, f32x4_t& s3, f32x4_t& s4, f32x4_t& s5, f32x4_t& s6, f32x4_t& s7,
                                             f32x4_t (&o)[4][NQ], int nq) {
  if (flag) {
    l *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      negm[i] -= delta;
      s0[i] -= delta; s1[i] -= delta; s2[i] -= delta; s3[i] -= delta;
      s4[i] -= delta; s5[i] -= delta; s6[i] -= delta; s7[i] -= delta;
      o[0][nq][i] *= alpha; o[1][nq][i] *= alpha; o[2][nq][i] *= alpha; o[3][nq][i] *= alpha;
    }
  }
}

// item: the tile of 256 query rows, numbered through the heads ((batch, head) * row_tiles + tile; rows at or beyond p.Sq
// do not exist); LOOP: the first one, the workgroup goes on with item + 32, item + 64, ... below `end`.  Otherwise the
// workgroup owns rows first_row .. first_row + part_rows of the tile.
// LDS: K stages at 0 and one tile, V stages behind them, with LOOP the output staging behind those; swizzles and operand
// layouts as in fa_fwd16_kernel (D 128) and fa_fwd16_d64_kernel (D 64: rows of 128 bytes, K chunk p of row r at
// p ^ ((r >> 1) & 7), V chunk p at p ^ ((r >> 1) & 3)).
template <int DT, bool LOOP, bool KEYMASK, int D>
__device__ __forceinline__ void fa16_flex_body(const FaParams& p, MSD_LDS char* smem, int item, int first_row, int part_rows,
                                               int end) {
  using E = Elem<DT>;
  using T = typename E::type;
  using X8 = typename E::x8;
  static_assert(D == 128 || (D == 64 && !LOOP), "head_dim");
  constexpr int NW = 8, BN = 128, NQ = LOOP ? 2 : 1;
  constexpr int kRowBytes = 2 * D, kDmaRows = 1024 / kRowBytes, NDB = D / 16, NKS = D / 32, kTileBytes = BN * kRowBytes;
  constexpr int NKB = BN / 16, NJ = BN / 32;  // 16-key blocks of the first product, 32-key steps of the second
  constexpr int kWaveRows = 16 * NQ;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  // the lane's number for the rarely run parts; LOOP, whose products need the registers: computed anew in each of them
  auto lane_here = [&]() __attribute__((always_inline)) {
    int l = lane;
    if constexpr (LOOP) {
      l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
      asm volatile("" : "+v"(l));
    }
    return l;
  };
  // (where the mask and head_dim 128 leave no vector register for spilled scalar ones; elsewhere a load of its own wait costs more)
  auto args_here = [&]() __attribute__((always_inline)) {
    if constexpr (KEYMASK && D == 128) return fa_args_here();
    else return &p;
  };
  const auto a0 = args_here();
  const int Sq = a0->Sq, Skv = a0->Skv;
  const float scale_log2 = a0->scale_log2;
  const int row_tiles = (Sq + 255) / 256;
  int b, n, row0;  // the tile at hand: batch entry, head, first query row of the wave
  auto locate = [&](auto a, int it, int& ib, int& in, int& irow) __attribute__((always_inline)) {
    const int bn = it / row_tiles, heads = a->N;
    ib = bn / heads;
    in = bn - ib * heads;
    irow = (it - bn * row_tiles) * 256 + first_row + wave * kWaveRows;
  };
  locate(a0, item, b, n, row0);
  const bool busy = LOOP || (wave * kWaveRows < part_rows && row0 < Sq);

  // ---- staging (LDS-DMA) -------------------------------------------------------------------------------------
  const int k_row_bytes = (int)a0->k_ss * 2, v_row_bytes = (int)a0->v_ss * 2;
  const int k_range = (int)(((long long)(Skv - 1) * a0->k_ss + D) * 2), v_range = (int)(((long long)(Skv - 1) * a0->v_ss + D) * 2);
  const T *kg, *vg;
  auto point_at_keys = [&](auto a, int ib, int in) __attribute__((always_inline)) {
    const int ikv = in / (a->N / a->Nkv);
    kg = (const T*)a->k + ib * a->k_sb + ikv * a->k_sn;
    vg = (const T*)a->v + ib * a->v_sb + ikv * a->v_sn;
  };
  point_at_keys(a0, b, n);
  int k_voff, v_voff;
  {
    const int row = kDmaRows * wave + lane / (kRowBytes / 16);  // groups of one wave lie kDmaRows * NW rows apart: same swizzles
    const int pc = lane % (kRowBytes / 16);
    const int ksw = D == 128 ? row & 15 : (row >> 1) & 7, vsw = D == 128 ? row & 7 : (row >> 1) & 3;
    k_voff = row * k_row_bytes + ((pc ^ ksw) << 4);
    v_voff = row * v_row_bytes + (((((pc >> 1) ^ vsw) << 1) | (pc & 1)) << 4);
  }
  auto load_tile = [&](int key0, int stage) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)kg, 0, k_range, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)vg, 0, v_range, 0x00020000);
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
  X8 qf[NQ][NKS];
  auto load_q = [&](auto a, int ib, int in, int irow) __attribute__((always_inline)) {
    const T* qg = (const T*)a->q + ib * a->q_sb + in * a->q_sn;
    const int ql = lane_here(), qc = ql & 15, qgr = ql >> 4;
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq) {
      const int qrow = irow + nq * 16 + qc;
      const T* src = qg + (long long)(qrow < Sq ? qrow : 0) * a->q_ss + 8 * qgr;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) qf[nq][ks] = *(const X8*)(src + 32 * ks);
    }
  };
  f32x4_t oacc[NDB][NQ], negm[NQ], lt[NQ];
  float l_run[NQ];
  X8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = E::from_float(1.f);

  // per-lane parts of the LDS read addresses
  unsigned k_lds[NKS], v_lds[4];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    k_lds[ks] = (unsigned)(uintptr_t)smem + c * kRowBytes + (((4 * ks + g) ^ (D == 128 ? c : c >> 1)) << 4);
#pragma unroll
  for (int db = 0; db < 4; ++db)
    v_lds[db] = (unsigned)(uintptr_t)smem + 2 * kTileBytes + (4 * g + (c >> 2)) * kRowBytes +
                ((db ^ (D == 128 ? 4 * (g & 1) + (c >> 2) : ((4 * g + (c >> 2)) >> 1) & 3)) << 5) + 8 * (c & 3);

  const int tiles = (Skv + BN - 1) / BN;
  load_q(a0, b, n, row0);
  load_tile(0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  bool first = true;

  // ---- key mask: words of visible keys of the current tile, bit l of word j = key 4 * l + j -----------------------------
  unsigned kvis[4] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu}, kraw = 0;
  const unsigned char* mask_g = nullptr;
  auto mask_request = [&](int key0) __attribute__((always_inline)) {
    if constexpr (KEYMASK) {
      kraw = 0;
      const int k4 = key0 + 4 * (lane_here() & (BN / 4 - 1));
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
      for (int j = 0; j < 4; ++j)  // (lanes 0 .. 31; the others hold the same bytes again)
        kvis[j] = (unsigned)__builtin_amdgcn_ballot_w64(((kraw >> (8 * j)) & 0xffu) != 0);
    }
  };

  // the products of the tile whose keys start at key0; next_mask0: first key of the mask bytes to request, < 0: none
  auto compute = [&](auto stage_c, const int key0, const int next_mask0) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_c)::value;
    const unsigned kv_all = kvis[0] & kvis[1] & kvis[2] & kvis[3];

    // S^T = K Q^T: operand groups of 2 key blocks of one 32-wide head_dim step, kAhead groups ahead of their use
    f32x4_t sacc[NKB][NQ];
    constexpr int kPer = NKB / 2, kGroups = NKS * kPer, kAhead = 3;
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
        for (int nq = 0; nq < NQ; ++nq)
          sacc[2 * qu + i][nq] =
              E::mfma16(afrag[gi % (kAhead + 1)][i], qf[nq][ks], ks == 0 ? negm[nq] : sacc[2 * qu + i][nq]);
    });
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
    for (int gi = 0; gi < kGroups - kAhead; ++gi) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * NQ, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2 * NQ * kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);

    if (key0 + BN > Skv) {  // keys past the end of the sequence (last tile only)
      const int g4 = 4 * (lane_here() >> 4);
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (key0 + 16 * kb + g4 + i >= Skv) {
#pragma unroll
            for (int nq = 0; nq < NQ; ++nq) sacc[kb][nq][i] = -INFINITY;
          }
    }
    if constexpr (KEYMASK) {
      if (kv_all != 0xffffffffu) {
        const int mg = lane_here() >> 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned w = kvis[i] >> mg;  // key 16 * kb + 4 * g + i is bit 4 * kb + g of word i
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
            if (!((w >> (4 * kb)) & 1u)) {
#pragma unroll
              for (int nq = 0; nq < NQ; ++nq) sacc[kb][nq][i] = -INFINITY;
            }
        }
      }
    }

    // online softmax (exp2 domain, lazily moved reference maximum; see fa_fwd_kernel)
    X8 pf[NQ][NJ];
    bool seen = !KEYMASK;
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq) {
      float mx = sacc[0][nq][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[kb][nq][i]);
      if constexpr (KEYMASK) seen = seen || __builtin_amdgcn_ballot_w64(mx > -INFINITY) != 0;
      float delta = 0.f, alpha = 1.f;
      int moved = 0;
      if (first || __builtin_amdgcn_ballot_w64(mx > kTau) != 0) {
        mx = quarter_max(mx);
        delta = first ? mx : fmaxf(mx, 0.f);
        delta = (delta == -INFINITY) ? 0.f : delta;
        // (first tile: sums and outputs are still zero; 2^-delta would overflow for rows far below zero and 0 * inf is NaN)
        alpha = first ? 1.f : fast_exp2(-delta);
        moved = 1;
      }
      l_run[nq] += lt[nq][0];
      fa16_rescale(__builtin_amdgcn_readfirstlane(moved), delta, alpha, l_run[nq], negm[nq], sacc[0][nq], sacc[1][nq],
                   sacc[2][nq], sacc[3][nq], sacc[4][nq], sacc[5][nq], sacc[6][nq], sacc[7][nq], oacc, nq);
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
    if (next_mask0 >= 0) mask_request(next_mask0);  // lands during the second product
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
        for (int nq = 0; nq < NQ; ++nq) oacc[4 * dbh + d4][nq] = E::mfma16(u.x, pf[nq][j], oacc[4 * dbh + d4][nq]);
      }
      if constexpr (dbh == 0) {
#pragma unroll
        for (int nq = 0; nq < NQ; ++nq)
          lt[nq] = E::mfma16(ones, pf[nq][j], j == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : lt[nq]);
      }
    });
    first = first && !seen;
  };
  // one key tile; next_key0: the first key of the tile to request (of the rows that kg and vg point at), < 0: none;
  // other_rows: it belongs to the workgroup's next tile of rows
  auto tile_step = [&](auto stage_c, const int key0, const int next_key0, const bool other_rows) __attribute__((always_inline)) {
    if (next_key0 >= 0) load_tile(next_key0, decltype(stage_c)::value ^ 1);
    if (busy) compute(stage_c, key0, other_rows ? -1 : next_key0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the next tile has landed
    mask_reduce();
    __syncthreads();
  };

  for (;;) {
    if constexpr (KEYMASK) {
      const auto a = args_here();
      mask_g = a->mask + b * a->m_sb + n * a->m_sn;
      mask_request(0);
      mask_reduce();
    }
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq) {
      const int qc = lane_here() & 15;
      const bool ok = row0 + nq * 16 + qc < Sq;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        X8 v = qf[nq][ks];
        if (!ok) v = X8{0};
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = E::from_float((float)v[j] * scale_log2);
        qf[nq][ks] = v;
      }
      l_run[nq] = 0.f;
      negm[nq] = lt[nq] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int db = 0; db < NDB; ++db) oacc[db][nq] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    first = true;
    const bool more = LOOP && item + 32 < end;
    int b_nx = 0, n_nx = 0, row0_nx = 0;
    unsigned touched = 0;
    if (LOOP && more) {
      const auto a = args_here();
      locate(a, item + 32, b_nx, n_nx, row0_nx);
      // a word of every 128-byte line of the next rows of q, so that they wait in the L2
      const int qrow = min(row0_nx + (lane_here() >> 1), Sq - 1);
      touched = *(const unsigned*)((const T*)a->q + b_nx * a->q_sb + n_nx * a->q_sn + (long long)qrow * a->q_ss + (lane_here() & 1) * 64);
    }
    for (int t = 0; t < tiles; t += 2) {
      tile_step(std::integral_constant<int, 0>{}, t * BN, t + 1 < tiles ? (t + 1) * BN : -1, false);
      if (t + 1 < tiles) {
        // (an even number of key tiles: the last step requests the first key tile of the next rows)
        const bool other_rows = LOOP && more && t + 2 >= tiles;
        if (other_rows) point_at_keys(args_here(), b_nx, n_nx);
        tile_step(std::integral_constant<int, 1>{}, (t + 1) * BN, t + 2 < tiles ? (t + 2) * BN : (other_rows ? 0 : -1), other_rows);
      }
    }
    if constexpr (LOOP) {
      asm volatile("" ::"v"(touched));
      if (more) {  // (an odd number: it goes into the stage of the last step, which no wave reads any more)
        load_q(args_here(), b_nx, n_nx, row0_nx);
        if (tiles & 1) {
          point_at_keys(args_here(), b_nx, n_nx);
          load_tile(0, 0);
        }
      }
    }

    // ---- normalise, transpose 16 rows at a time through LDS (16-byte chunk k of row r at chunk k ^ r), coalesced store ------
    // LOOP: behind the tile stages, which already fill with the next rows' keys; otherwise in them: no wave reads them any more
    if (busy) {
      constexpr int kChunks = D / 8, kSwz = kChunks - 1;
      const auto a = args_here();
      T* og = (T*)a->o + b * a->o_sb + n * a->o_sn;
      float* lse = a->lse ? a->lse + ((long long)b * a->N + n) * Sq : nullptr;
      const long long o_ss = a->o_ss;
      MSD_LDS char* ost = smem + (LOOP ? 4 * kTileBytes : 0) + wave * 16 * kRowBytes;
      const int ol = lane_here(), oc = ol & 15, ogr = ol >> 4;
#pragma unroll
      for (int nq = 0; nq < NQ; ++nq) {
        const float l_tot = l_run[nq] + lt[nq][0];
        const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        const int qrow_l = row0 + nq * 16 + oc;
        if (lse && ogr == 0 && qrow_l < Sq)
          lse[qrow_l] = l_tot > 0.f ? -negm[nq][0] * 0.6931471805599453f + __logf(l_tot) : -INFINITY;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          typename E::x4 pk;
#pragma unroll
          for (int i = 0; i < 4; ++i) pk[i] = E::from_float(oacc[db][nq][i] * inv);
          *(MSD_LDS typename E::x4*)(ost + oc * kRowBytes + (((2 * db + (ogr >> 1)) ^ (oc & kSwz)) << 4) + 8 * (ogr & 1)) = pk;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < kChunks / 4; ++i) {
          const int row = i * (64 / kChunks) + ol / kChunks, ch = ol % kChunks, qrow = row0 + nq * 16 + row;
          const i32x4_t v = *(MSD_LDS const i32x4_t*)(ost + row * kRowBytes + ((ch ^ (row & kSwz)) << 4));
          if (qrow < Sq) *(i32x4_t*)(og + (long long)qrow * o_ss + ch * 8) = v;
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    if constexpr (LOOP) {
      if (!more) return;
      item += 32;
      b = b_nx;
      n = n_nx;
      row0 = row0_nx;
      if (tiles & 1) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        __syncthreads();
      }
    } else {
      return;
    }
  }
}
#endif

}  // namespace msd
