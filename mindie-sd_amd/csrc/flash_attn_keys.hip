// Dense attention over at most 256 keys at head_dim 128 for gfx950 (MI355X): the video tokens' attention over a short text.
//
// The keys of a (batch, head) fit a CU's LDS whole (K and V of 256 keys: 128 KiB), so a workgroup stages them once and its eight
// waves then go through the head's query rows 32 at a time, each at its own pace: nothing is staged again, no barrier is met
// until the head changes, and while one wave waits for its queries or stores its output the other waves of the SIMD multiply.
// With all scores of 32 rows in registers the softmax is the plain one: the row's maximum, no running sums to rescale.
// Operand layouts, LDS swizzles and the transposed formulation are those of fa_fwd16_kernel (flash_attn_fwd.hip): lane
// (c = lane % 16, g = lane / 16) owns query columns 16 * nq + c, S^T blocks of 16 keys come from one 16-byte K read, V^T from
// transposing reads.
//
// What bounds it: up to 128 keys reading Q and writing O (40 heads x 32760 queries x 128 keys 154 us, 676 MB behind the L2 = 4.4 TB/s,
// the matrix pipe busy 25 % of the cycles), beyond that the products and the LDS reads behind them, every wave all keys for its 32
// rows, and at 7 and 8 blocks the wait for queries that are not requested ahead (256 keys 204 us, 0.84 PFLOP/s, 41 %).  Against the 4-wave
// kernel, which stages every key tile for each 128 rows: 40 heads x 32760 queries over 64 / 91 / 128 / 188 / 226 / 256 keys 160 / 177 /
// 176 / 221 / 253 / 251 -> 154 / 155 / 156 / 168 / 200 / 204 us, 16 x 19666 33 / 41 / 41 / 50 / 57 / 57 -> 29 / 32 / 34 / 42 / 47 / 48 us,
// 16 x 5000 13.6 / 16.3 / 16.1 / 19.2 / 21.1 / 21.2 -> 11.9 / 12.8 / 13.9 / 16.4 / 18.0 / 18.2 us.  At most 64 keys (one key tile there)
// over more than a million rows are the same copy of Q to O in both: 0.95 (2 x 12 heads x 60000) to 1.14 (8 x 40 x 4096), by heads and
// layout.  Error against 64 bits 0.98 to 1.00 of that kernel's (no rescaling).  Vector registers: 160 with one block of 32 keys, 219 to
// 246 with more, none spilled; scalar ones spilled 3 (two blocks) to 22 (eight), outside of the loop over the rows.
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "fa_params.hpp"

namespace msd {

constexpr int kKeysWaves = 8, kKeysRows = 32;  // waves of a workgroup, query rows of a wave at a time

#if defined(__HIP_DEVICE_COMPILE__)
// first of the units (32 query rows each, numbered through the heads) of workgroup (x, j): every XCD has a run of consecutive
// units, every workgroup a run of its XCD's, equal up to one unit
__device__ __forceinline__ int keys_first_unit(int units, int x, int j, int per_xcd) {
  const int a = (int)((long long)units * x / 8), b = (int)((long long)units * (x + 1) / 8);
  return a + (int)((long long)(b - a) * j / per_xcd);
}
#endif

// NJ: 32-key blocks
template <int DT, int NJ>
__global__ __launch_bounds__(kKeysWaves * 64, 1) void fa16_keys_kernel(const FaParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  using E = Elem<DT>;
  using T = typename E::type;
  using X8 = typename E::x8;
  constexpr int kRowBytes = 256, NKB = 2 * NJ, kKeys = 32 * NJ, kV = kKeys * kRowBytes;  // V behind K
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  MSD_LDS char* smem = (MSD_LDS char*)smem_raw;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row_units = (p.Sq + kKeysRows - 1) / kKeysRows, units = p.B * p.N * row_units, per_xcd = gridDim.x >> 3;
  int unit = keys_first_unit(units, blockIdx.x & 7, blockIdx.x >> 3, per_xcd);
  const int unit_end = keys_first_unit(units, blockIdx.x & 7, (blockIdx.x >> 3) + 1, per_xcd);

  const int k_row_bytes = (int)p.k_ss * 2, v_row_bytes = (int)p.v_ss * 2;
  int k_voff, v_voff;  // the lane's 16 bytes of a 4-row group (1 KiB) of its wave; groups lie 32 rows apart: same swizzles
  {
    const int row = 4 * wave + (lane >> 4), pc = lane & 15;
    k_voff = row * k_row_bytes + ((pc ^ (row & 15)) << 4);
    v_voff = row * v_row_bytes + (((((pc >> 1) ^ (row & 7)) << 1) | (pc & 1)) << 4);
  }
  unsigned k_lds[4], v_lds[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) k_lds[ks] = (unsigned)(uintptr_t)smem + c * kRowBytes + (((4 * ks + g) ^ c) << 4);
#pragma unroll
  for (int db = 0; db < 4; ++db)
    v_lds[db] = (unsigned)(uintptr_t)smem + kV + (4 * g + (c >> 2)) * kRowBytes + ((db ^ (4 * (g & 1) + (c >> 2))) << 5) + 8 * (c & 3);
  MSD_LDS char* ost = smem + 2 * kV + wave * 16 * kRowBytes;
  X8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = E::from_float(1.f);

  for (bool again = false; unit < unit_end; again = true) {  // one (batch, head) after another
    const int bn = unit / row_units, b = bn / p.N, n = bn - b * p.N, nkv = n / (p.N / p.Nkv);
    const int seg_end = min(unit_end, (bn + 1) * row_units);
    if (again) __syncthreads();  // every wave has done with the head before
    {
      const T* kg = (const T*)p.k + b * p.k_sb + nkv * p.k_sn;
      const T* vg = (const T*)p.v + b * p.v_sb + nkv * p.v_sn;
      // (rows past the keys lie beyond the range and read as zeros)
      const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          (void*)kg, 0, (int)(((long long)(p.Skv - 1) * p.k_ss + 128) * 2), 0x00020000);
      const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          (void*)vg, 0, (int)(((long long)(p.Skv - 1) * p.v_ss + 128) * 2), 0x00020000);
#pragma unroll
      for (int i = 0; i < NJ; ++i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rsrc, (MSD_LDS void*)(smem + (i * 8 + wave) * 1024), 16, k_voff,
                                                 i * 32 * k_row_bytes, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rsrc, (MSD_LDS void*)(smem + kV + (i * 8 + wave) * 1024), 16, v_voff,
                                                 i * 32 * v_row_bytes, 0, 0);
      }
    }
    const T* qg = (const T*)p.q + b * p.q_sb + n * p.q_sn;
    T* og = (T*)p.o + b * p.o_sb + n * p.o_sn;
    X8 qf[2][4], qn[2][4];  // the rows at hand, and the next ones as they come from memory
    auto load_q = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int nq = 0; nq < 2; ++nq) {
        const int row = (u - bn * row_units) * kKeysRows + nq * 16 + c;
        const T* src = qg + (long long)min(row, p.Sq - 1) * p.q_ss + 8 * g;  // (rows past the end: computed, never stored)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qn[nq][ks] = *(const X8*)(src + 32 * ks);
      }
    };
    int u = unit + wave;
    constexpr bool kNext = NJ <= 6;  // the next rows' queries in registers meanwhile (7 and 8: no room for them)
    if (kNext && u < seg_end) load_q(u);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    for (; u < seg_end; u += kKeysWaves) {
      const int row0 = (u - bn * row_units) * kKeysRows;
      if (!kNext) load_q(u);
#pragma unroll
      for (int nq = 0; nq < 2; ++nq)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int j = 0; j < 8; ++j) qf[nq][ks][j] = E::from_float((float)qn[nq][ks][j] * p.scale_log2);
      if (kNext && u + kKeysWaves < seg_end) load_q(u + kKeysWaves);
      __builtin_amdgcn_sched_barrier(0);

      // ---- S^T = K Q^T: operand groups of 2 key blocks of one 32-wide head_dim step, kAhead groups ahead of their use ----------
      f32x4_t sacc[NKB][2];
      constexpr int kGroups = 4 * NJ, kAhead = 3;
      X8 afrag[kAhead + 1][2];
      auto k_read = [&](auto gi_c, X8(&dst)[2]) __attribute__((always_inline)) {
        constexpr int gi = decltype(gi_c)::value, ks = gi / NJ, qu = gi % NJ;
#pragma unroll
        for (int i = 0; i < 2; ++i) dst[i] = *(MSD_LDS const X8*)(uintptr_t)(k_lds[ks] + (2 * qu + i) * 16 * kRowBytes);
      };
      static_for<kAhead>([&](auto gi_c) __attribute__((always_inline)) { k_read(gi_c, afrag[decltype(gi_c)::value]); });
      static_for<kGroups>([&](auto gi_c) __attribute__((always_inline)) {
        constexpr int gi = decltype(gi_c)::value, ks = gi / NJ, qu = gi % NJ;
        if constexpr (gi + kAhead < kGroups) k_read(std::integral_constant<int, gi + kAhead>{}, afrag[(gi + kAhead) % (kAhead + 1)]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int nq = 0; nq < 2; ++nq)
            sacc[2 * qu + i][nq] = E::mfma16(afrag[gi % (kAhead + 1)][i], qf[nq][ks],
                                             ks == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : sacc[2 * qu + i][nq]);
      });
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
      for (int gi = 0; gi < kGroups - kAhead; ++gi) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * kAhead, 0);
      __builtin_amdgcn_sched_barrier(0);

      if (p.Skv != kKeys) {  // keys past the end: in the last 32 only
#pragma unroll
        for (int kb = NKB - 2; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * kb + 4 * g + i >= p.Skv) sacc[kb][0][i] = sacc[kb][1][i] = -INFINITY;
      }

      // ---- softmax of the rows (exp2 domain; the scale went into Q) ------------------------------------------------------
      X8 pf[2][NJ];
      float m[2];
#pragma unroll
      for (int nq = 0; nq < 2; ++nq) {
        float mx = sacc[0][nq][0];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[kb][nq][i]);
        mx = quarter_max(mx);
        m[nq] = mx == -INFINITY ? 0.f : mx;  // (no finite score: sums of zero, as with a running maximum)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            pf[nq][j][t] = E::from_float(fast_exp2(sacc[2 * j][nq][t] - m[nq]));
            pf[nq][j][4 + t] = E::from_float(fast_exp2(sacc[2 * j + 1][nq][t] - m[nq]));
          }
      }

      // ---- O^T = V^T P^T: steps of (32 keys) x (4 head_dim blocks), V^T fragments requested one step ahead; row sums as
      // ones x P^T ----------------------------------------------------------------------------------------------------------
      f32x4_t oacc[8][2], l[2];
      s16x4_t vf[2][8];
      auto issue = [&](auto step_c, s16x4_t(&dst)[8]) __attribute__((always_inline)) {
        constexpr int s = decltype(step_c)::value, off = 32 * (s >> 1) * kRowBytes;
#pragma unroll
        for (int d4 = 0; d4 < 4; ++d4) {
          const unsigned a = v_lds[d4] ^ ((s & 1) << 7);
          dst[2 * d4] = lds_read_tr16_async<off>(a);
          dst[2 * d4 + 1] = lds_read_tr16_async<off + 16 * kRowBytes>(a);
        }
      };
      issue(std::integral_constant<int, 0>{}, vf[0]);
      static_for<2 * NJ>([&](auto step_c) __attribute__((always_inline)) {
        constexpr int s = decltype(step_c)::value, j = s >> 1, dbh = s & 1;
        if constexpr (s + 1 < 2 * NJ) {
          issue(std::integral_constant<int, s + 1>{}, vf[(s + 1) & 1]);
          lds_wait_tr<8>(vf[s & 1]);
        } else {
          lds_wait_tr<0>(vf[s & 1]);
        }
#pragma unroll
        for (int d4 = 0; d4 < 4; ++d4) {
          union { s16x4_t s2[2]; X8 x; } v;
          v.s2[0] = vf[s & 1][2 * d4];
          v.s2[1] = vf[s & 1][2 * d4 + 1];
#pragma unroll
          for (int nq = 0; nq < 2; ++nq)
            oacc[4 * dbh + d4][nq] = E::mfma16(v.x, pf[nq][j], j == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : oacc[4 * dbh + d4][nq]);
        }
        if constexpr (dbh == 0) {
#pragma unroll
          for (int nq = 0; nq < 2; ++nq) l[nq] = E::mfma16(ones, pf[nq][j], j == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : l[nq]);
        }
      });

      // ---- normalise, transpose 16 rows at a time through the wave's 4 KiB (16-byte chunk k of row r at chunk k ^ r), store ------
#pragma unroll
      for (int nq = 0; nq < 2; ++nq) {
        const float l_tot = l[nq][0], inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        const int qrow = row0 + nq * 16 + c;
        if (p.lse && g == 0 && qrow < p.Sq)
          p.lse[((long long)b * p.N + n) * p.Sq + qrow] = l_tot > 0.f ? m[nq] * 0.6931471805599453f + __logf(l_tot) : -INFINITY;
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          typename E::x4 pk;
#pragma unroll
          for (int i = 0; i < 4; ++i) pk[i] = E::from_float(oacc[db][nq][i] * inv);
          *(MSD_LDS typename E::x4*)(ost + c * kRowBytes + (((2 * db + (g >> 1)) ^ c) << 4) + 8 * (g & 1)) = pk;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = i * 4 + g, row = row0 + nq * 16 + r;
          const i32x4_t v = *(MSD_LDS const i32x4_t*)(ost + r * kRowBytes + ((c ^ r) << 4));
          if (row < p.Sq) *(i32x4_t*)(og + (long long)row * p.o_ss + c * 8) = v;
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    unit = seg_end;
  }
#endif
}

template <int DT>
static int launch_keys(const FaParams& p, hipStream_t stream) {
  auto launch = [&](auto nj_c) -> int {
    constexpr int NJ = decltype(nj_c)::value;
    constexpr int kLds = NJ * 32 * 512 + kKeysWaves * 16 * 256;
    auto kern = fa16_keys_kernel<DT, NJ>;
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return MSD_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3(kCus), dim3(kKeysWaves * 64), kLds, stream, p);
    return hipGetLastError() == hipSuccess ? MSD_OK : MSD_ERR_LAUNCH;
  };
  switch ((p.Skv + 31) / 32) {
    case 1: return launch(std::integral_constant<int, 1>{});
    case 2: return launch(std::integral_constant<int, 2>{});
    case 3: return launch(std::integral_constant<int, 3>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    case 5: return launch(std::integral_constant<int, 5>{});
    case 6: return launch(std::integral_constant<int, 6>{});
    case 7: return launch(std::integral_constant<int, 7>{});
    default: return launch(std::integral_constant<int, 8>{});
  }
}

// Where it pays: keys that fit (256), 8 units to every workgroup (fewer leave waves without rows; 1024 units, 8 heads x 4096, 256
// keys 12.0 against 12.2 us, 840 units, 24 heads x 1100, 12.0 against 14.9), and heads long enough for their keys to be staged
// alone (512 rows: 35 -> 34 us at 8 x 40 heads, 256 keys; 256 rows: 43 against 50, 128 rows: 35 against 47 us).
bool fa16_keys_preferred(const FaParams& p) {
  const long long units = (long long)p.B * p.N * ((p.Sq + kKeysRows - 1) / kKeysRows);
  return p.Skv <= 256 && p.Sq >= 512 && units >= 8 * kCus && units < (1ll << 30);
}

int launch_fa16_keys(const FaParams& p, int dtype, hipStream_t stream) {
  return dtype == MSD_DTYPE_BF16 ? launch_keys<MSD_DTYPE_BF16>(p, stream) : launch_keys<MSD_DTYPE_F16>(p, stream);
}

}  // namespace msd
