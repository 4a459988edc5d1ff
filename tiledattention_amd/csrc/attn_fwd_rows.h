// SDPA forward for CDNA4 (gfx950), fp32 accumulation: small independent workgroups, several
// on a CU (compiled into attn_fwd_wide.hsaco).
//
// Math: the reference's tiled forward with fp32 accumulation
// (src/tiledattention/kernels/flash_fwd.py:374-446).
//
// * A workgroup is four waves and 128 query rows; wave w owns rows [32 w, 32 w + 32) and
//   walks every key of them itself, so no state is shared and nothing is merged at the end.
// * Keys come in tiles of 64, HBM -> LDS directly, two stages each of K and V; one barrier a
//   tile (the loads of tile t + 1 go out right after it, into the stage tile t - 1 left).
// * Two to four such workgroups share a CU (registers and LDS), in no fixed phase to one
//   another: one's softmax and loads run beside another's matrix products.
// * Operand layouts, swizzles and the lazy rescale are the eight-wave kernel's
//   (attn_fwd_pp.hip).
//
// It runs the grids of short rows and many heads, where the eight-wave kernel's workgroup, one
// a CU, spends as long on its prologue, pipeline fill and merge as on its keys.  Back-to-back
// launches of both on one card: B32 H12 S197 D64 fp16 non-causal 16.0 -> 13.2 us, B16 H16 S512 D64
// bf16 31.4 -> 25.7, B64 H12 S128 D64 fp16 causal 20.2 -> 11.1, B8 H32 S320 D128 bf16 31.3 -> 26.7
// (their 39, 67, 75 and 84 MB of q, k, v and o take 7.4, 12.8, 14.4 and 16 us at a large copy's rate).  Long rows reach what the
// eight-wave kernels do at D = 64 and less at 128 (B4 H16 S4096: 278 us against 265, 482 against
// 427), and few blocks lose (B1 H8 S8192 D64 causal 102 against 76).  64 query rows a wave, which
// halves the LDS operand reads, was not faster (12.4 -> 14.1, 24.3 -> 24.4 us), nor were eight
// waves a workgroup in general, or a raised priority for either kind of work; without any
// softmax arithmetic the four cases above take 10-12 % less, so loads and latency bound them.
// A second copy of the tile for a last one of at most 32 keys (bit-identical) was faster where such
// rows are short (B64 H12 S80 D64 9.5 -> 8.9 us, B32 H12 S197 14.2 -> 13.7), but the copy itself costs
// every other row 2-4 % (S250 14.7 -> 15.3, D96 S1000 58.3 -> 60.6, causal D64 S512 21.7 -> 22.2) and
// the input-dtype kernels spill with it.
//
// Input-dtype accumulation (LOWP_TN): the same workgroups with the eight-wave kernel's two key
// slices a row, both in one wave (even and odd tiles), so results and errors are the same to the
// merge's last bit (2-norm 1e-5): B4 H16 S4096 D64 fp16 430 -> 369 us, bf16 430 -> 352;
// B16 H16 S512 fp16 44 -> 30.  VALU-bound (84 % of cycles): per tile and lane 32 FMAs, 32
// exponentials, 32 sums, 16 maxima, 16 packs, the rounding of O (48) and its rescale (32, three
// tiles in five).  The rescale is a branch of its own in front of one rounding: a branch with a
// rounding on either side kept a second copy of O alive (7-13 registers spilled at D = 64, over
// 100 at 128).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "attn_fwd_common.h"
#include "attn_fwd_params.h"
#include "attn_fwd_split.h"

namespace ta {

constexpr int kRowsKeys = 64;  // keys per tile
constexpr int kRowsWaves = 4;
constexpr int kRowsExact = 3;  // tiles whose largest P is exact
constexpr float kRowsFar = 32.0f;  // a tile that far (log2) below the point keeps the point

// p.n_qblk = ceil(S / 128).
template <int DT, int D, bool CAUSAL, bool TAIL, int LOWP_TN = 0>
__device__ __forceinline__ void attn_fwd_rows_body(const FwdParams& p) {
  static_assert(D == 64 || D == 96 || D == 128 || D == 160, "head dims 64, 96, 128 and 160");
  constexpr int NW = kRowsWaves;
  // Input-dtype accumulation: two key slices a row, the even and the odd tiles, each with its
  // own (m, l, O): the slices, the arithmetic and the cadence of rounding (once per TILE_N keys
  // of a slice) of the eight-wave kernel's two wave groups.
  constexpr bool LOWP = LOWP_TN != 0;
  constexpr int NSL = LOWP ? 2 : 1;
  static_assert(LOWP_TN == 0 || LOWP_TN == 64 || LOWP_TN == 128, "TILE_N");
  constexpr int TK = kRowsKeys;
  constexpr int TM = 32 * NW;
  constexpr int RB = 2 * D;              // bytes per key row
  constexpr int STAGE = TK * RB;
  constexpr int CPR = D / 8;             // 16-byte chunks per row
  constexpr bool kPow2 = D == 64 || D == 128;  // 1 KiB of LDS is whole rows
  constexpr int NLD = STAGE / 1024 / NW; // loads per wave per tensor per tile
  constexpr int DK = D / 16;
  constexpr int DB = D / 32;
  constexpr int KB = TK / 32;
  static_assert(STAGE % (1024 * NW) == 0 && NW % 4 == 0, "the stage splits over the waves");
  using DTy = DType<DT>;
  __shared__ __attribute__((aligned(1024))) char lds_k0[STAGE];
  __shared__ __attribute__((aligned(1024))) char lds_k1[STAGE];
  __shared__ __attribute__((aligned(1024))) char lds_v0[STAGE];
  __shared__ __attribute__((aligned(1024))) char lds_v1[STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hl = lane >> 5;

  const WorkItem wi = whole_item(blockIdx.x, p.n_bh, p.n_qblk, p.sched, CAUSAL, CAUSAL ? p.head_group : 0);
  const int S = p.S;
  const int b = wi.bh / p.H;
  const int h = wi.bh - b * p.H;
  const uint16_t* __restrict__ qp = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* __restrict__ kp = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* __restrict__ vp = p.v + b * p.v_sb + h * p.v_sh;
  uint16_t* __restrict__ op = p.o + b * p.o_sb + h * p.o_sh;
  const int k_rb = (int)p.k_ss * 2;
  const int v_rb = (int)p.v_ss * 2;
  const int d_real = p.d_real;
  const float c = p.scale_log2;

  const int q0 = wi.qt * TM;
  const int wq0 = q0 + 32 * wave;
  const int my_q = wq0 + l32;
  const int n_tiles = ((CAUSAL ? min(S, q0 + TM) : S) + TK - 1) / TK;
  // keys this wave needs (none when its rows are all past S)
  const int wave_kv_end = TAIL && wq0 >= S ? 0 : CAUSAL ? min(S, wq0 + 32) : S;

  // ---- loads: wave w fills the 1 KiB pieces w + NW i of a stage; lane l of piece g writes the
  // stage's 16-byte chunk 64 g + l, physical chunk (64 g + l) % CPR of row (64 g + l) / CPR.
  // Logical chunks at or past d_real read as zero (attn_fwd_pp.hip).  Swizzles: D = 64 and 128
  // as there; rows of 12 or 20 chunks (D = 96, 160) start at a multiple of 4 of the 16 bank
  // units that moves on by 12 or 4 a row, so four rows in a row already read V's 64 bytes
  // without conflict, and K's 16 rows do with the chunk's low two bits ^ (row >> 2) & 3.
  constexpr int kZeroChunk = INT32_MIN;
  constexpr int NVO = kPow2 ? 1 : NLD;  // whole rows: every piece of a wave is one offset apart
  int kvo[NVO], vvo[NVO];
#pragma unroll
  for (int i = 0; i < NVO; ++i) {
    const int ch = (wave + NW * i) * 64 + lane;
    const int row = ch / CPR, pc = ch % CPR;
    const int lck = pc ^ (kPow2 ? pp_swz_k<D>(row) : (row >> 2) & 3);
    const int lcv = pc ^ (kPow2 ? pp_swz_v<D>(row) : 0);
    kvo[i] = 8 * lck < d_real ? row * k_rb + (lck << 4) : kZeroChunk;
    vvo[i] = 8 * lcv < d_real ? row * v_rb + (lcv << 4) : kZeroChunk;
  }
  auto dma = [&](const uint16_t* gbase, int64_t row_stride, int rb, const int* vo, int t, char* stage) {
    const int row0 = t * TK;
    const __amdgpu_buffer_rsrc_t r = row_rsrc(gbase + (int64_t)row0 * row_stride, S - row0, rb);
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, (__attribute__((address_space(3))) void*)(stage + (wave + NW * i) * 1024), 16,
          kPow2 ? vo[0] + i * NW * (1024 / RB) * rb : vo[i], 0, 0, 0);
    }
  };

  // ---- LDS reads (attn_fwd_pp.hip) -----------------------------------------------------
  const int mk = kPow2 ? pp_swz_k<D>(l32) : (l32 >> 2) & 3;
  const int k_rd = l32 * RB + (kPow2 ? 32 * (mk >> 1) : 0) + 16 * (hl ^ (mk & 1));
  const int k_odd = 32 * (mk >> 1);  // D = 96, 160: bit 1 of the chunk is (kk & 1) ^ (mk >> 1)
  auto k_col = [&](int kk) {
    return kPow2 ? k_rd ^ (32 * kk) : k_rd + (kk & 1 ? 32 - k_odd : k_odd) + 64 * (kk >> 1);
  };
  const int tr_r = (lane & 15) >> 2;
  const int tr_d = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int v_rd = (4 * hl + tr_r) * RB + 16 * ((tr_d >> 3) ^ (kPow2 ? pp_swz_v<D>(4 * hl + tr_r) : 0)) + 2 * (tr_d & 7);
  auto v_col = [&](int db) { return kPow2 ? v_rd ^ (64 * db) : v_rd + 64 * db; };

  // ---- Q fragment: lane l holds row wq0 + l % 32, columns 16 kk + 8 (l / 32) .. + 8
  u32x4 qf[DK];
  float m_sl[NSL], l_sl[NSL];
  f32x16 o_sl[NSL][DB];
#pragma unroll
  for (int i = 0; i < NSL; ++i) {
    m_sl[i] = kNegLarge;
    l_sl[i] = 0.0f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o_sl[i][db] = f32x16{};
  }

  dma(kp, p.k_ss, k_rb, kvo, 0, lds_k0);
  dma(vp, p.v_ss, v_rb, vvo, 0, lds_v0);
  {
    const bool ok = my_q < S;
    const uint16_t* qrow = qp + (int64_t)(ok ? my_q : 0) * p.q_ss;
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
      const int d0 = 16 * kk + 8 * hl;
      qf[kk] = ok && d0 < d_real ? *(const u32x4*)(qrow + d0) : u32x4{0u, 0u, 0u, 0u};
    }
  }

  auto tile = [&](int t, const char* kst, const char* vst, auto par_tag) {
    constexpr int SL = LOWP ? decltype(par_tag)::value : 0;
    float& m_run = m_sl[SL];
    float& l_part = l_sl[SL];
    f32x16(&o_acc)[DB] = o_sl[SL];
    const int k0 = t * TK;
    if (k0 >= wave_kv_end) return;
    f32x16 s[KB];
    uint32_t pk[KB][8];
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
        const u32x4 a = *(const u32x4*)(kst + bk * 32 * RB + k_col(kk));
        s[bk] = DTy::mfma(a, qf[kk], kk == 0 ? f32x16{} : s[bk]);
      }
    }
    if ((CAUSAL && k0 + TK - 1 > wq0) || (TAIL && k0 + TK > S)) {
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * bk + (r >> 2) * 8 + hl * 4 + (r & 3);
          bool bad = false;
          if (CAUSAL) bad = key > my_q;
          if (TAIL) bad = bad || key >= S;
          s[bk][r] = bad ? kMasked : s[bk][r];
        }
      }
    }
    auto row_max = [&]() {
      float mxa = kMasked, mxb = kMasked;
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          mxa = vmax3_step(mxa, s[bk][r], s[bk][r + 1]);
          mxb = vmax3_step(mxb, s[bk][r + 2], s[bk][r + 3]);
        }
      }
      float a0, a1;
      swap32(vmax(mxa, mxb), a0, a1);
      return vmax(a0, a1);
    };
    if constexpr (LOWP) {
      // Exact running max; P from it, packed for P.V; l from the unrounded P; the products
      // accumulated since the last rounding rounded to the input dtype, rescaled first where
      // a row's max moved (attn_fwd_pp.hip).
      const float m_new = vmax(m_run, row_max());
      const float alpha = fast_exp2((m_run - m_new) * c);
      m_run = m_new;
      const float mc = m_run * c;
      float l4[4];
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float p0 = fast_exp2(__builtin_fmaf(s[bk][r], c, -mc));
          const float p1 = fast_exp2(__builtin_fmaf(s[bk][r + 1], c, -mc));
          pk[bk][r >> 1] = DTy::pack(p0, p1);
          const int j = (r >> 1) & 3;
          l4[j] = bk == 0 && r < 8 ? p0 + p1 : l4[j] + (p0 + p1);
        }
      }
      l_part = l_part * alpha + ((l4[0] + l4[1]) + (l4[2] + l4[3]));
      const bool moved = __ballot(!(alpha == 1.0f)) != 0;
      const float al = DTy::round(alpha);
      const bool round_now = LOWP_TN == 64 || ((t >> 1) & 1);  // step t >> 1 of the slice
      if (moved) {
#pragma unroll
        for (int db = 0; db < DB; ++db) o_acc[db] *= al;
      }
      if (round_now) {
#pragma unroll
        for (int db = 0; db < DB; ++db) {
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            // (kept packed: fp16 would otherwise be converted value by value, four
            // instructions a pair instead of three)
            uint32_t w = DTy::pack(o_acc[db][r], o_acc[db][r + 1]);
            asm("" : "+v"(w));
            o_acc[db][r] = DTy::lo(w);
            o_acc[db][r + 1] = DTy::hi(w);
          }
        }
      }
    }
    auto make_p = [&](float mc) {
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          pk[bk][r >> 1] = DTy::pack(fast_exp2(__builtin_fmaf(s[bk][r], c, -mc)),
                                     fast_exp2(__builtin_fmaf(s[bk][r + 1], c, -mc)));
        }
      }
      float l4[4];
#pragma unroll
      for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const int j = (r >> 1) & 3;
          l4[j] = bk == 0 && r < 8 ? DTy::sum2_head(pk[bk][r >> 1]) : DTy::sum2(pk[bk][r >> 1], l4[j]);
        }
      }
      return (l4[0] + l4[1]) + (l4[2] + l4[3]);
    };
    // Reference point of P: over the first kRowsExact tiles (O and l are zero at the first: nothing
    // to rescale) every tile's largest P is an exact power of two and carries no rounding: the
    // tile's own max where that is above the point so far, else whole log2 units above that max and
    // less than one below the point, so that O and l less than double.  That is as exact as the
    // eight-wave kernel, whose two key halves have a max each.  From then on the lazy rule of that
    // kernel (the max is reduced only where some lane's sum of P reaches the bound).
    // Against 64 bits, the eight-wave kernel's error = 1 (B H 264-384, N(0, 1), both dtypes):
    // with the running max instead S96 to S113 1.014-1.016, S128 1.013, causal to S200
    // 1.002-1.003; every further exact tile costs 1 % of the time.
    // (m_run is in log2 units here, score times c.)
    if constexpr (!LOWP) {
      if (t < kRowsExact) {
        const float mx = vmax(row_max() * c, m_run - kRowsFar);
        const float m_new = mx + vmax(__builtin_floorf(m_run - mx), 0.0f);
        if (t > 0 && __ballot(!(m_new == m_run))) {
          const float alpha = fast_exp2(m_run - m_new);
#pragma unroll
          for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
          l_part *= alpha;
        }
        m_run = m_new;
      }
      float l_step = make_p(m_run);
      if (t >= kRowsExact && __ballot(!(l_step < kRescaleBound))) {
        const float mx = row_max() * c;
        const bool need = mx - m_run > kRescaleLog2;
        if (__ballot(need)) {
          const float m_new = need ? mx : m_run;
          const float alpha = fast_exp2(m_run - m_new);
          m_run = m_new;
#pragma unroll
          for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
          l_part *= alpha;
          l_step = make_p(m_run);
        }
      }
      l_part += l_step;
    }
#pragma unroll
    for (int bk = 0; bk < KB; ++bk) {
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const u32x4 bfrag = {pk[bk][4 * kc + 0], pk[bk][4 * kc + 1], pk[bk][4 * kc + 2], pk[bk][4 * kc + 3]};
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const char* a0p = vst + v_col(db) + (32 * bk + 16 * kc) * RB;
          s16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)a0p);
          s16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a0p + 8 * RB));
          u32x2 w0 = __builtin_bit_cast(u32x2, r0);
          u32x2 w1 = __builtin_bit_cast(u32x2, r1);
          o_acc[db] = DTy::mfma(u32x4{w0[0], w0[1], w1[0], w1[1]}, bfrag, o_acc[db]);
        }
      }
    }
  };

  // Tile t: this wave's loads of it (issued a tile ago) have landed, then the barrier: every
  // wave's have, and every wave is done reading tile t - 1, whose stage takes tile t + 1.
  auto step = [&](int t, char* k_cur, char* v_cur, char* k_nxt, char* v_nxt, auto par_tag) {
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < n_tiles) {
      dma(kp, p.k_ss, k_rb, kvo, t + 1, k_nxt);
      dma(vp, p.v_ss, v_rb, vvo, t + 1, v_nxt);
    }
    tile(t, k_cur, v_cur, par_tag);
  };
  // The loop starts at a multiple of 32 bytes, whatever the prologue's length: D = 64 non-causal
  // B8 H12 S448 11.4 us here, 11.6 twenty bytes further on (S320 1.3 %, S512 1 %).
  asm volatile(".p2align 5");
  for (int t = 0; t < n_tiles; t += 2) {
    step(t, lds_k0, lds_v0, lds_k1, lds_v1, std::integral_constant<int, 0>{});
    if (t + 1 < n_tiles) step(t + 1, lds_k1, lds_v1, lds_k0, lds_v0, std::integral_constant<int, 1>{});
  }

  // ---- O = acc / l: the lane pair l, l + 32 holds halves of a row's 16-byte chunks; swapping
  // chunk g's upper half with chunk g + 1's lower half gives each lane a whole chunk.
  // (Input-dtype accumulation: the slices combined in fp32 and rounded to the input dtype, then
  // rnd(acc rnd(1 / l)).)
  f32x16(&o_acc)[DB] = o_sl[0];
  float la, lb, a0 = 1.0f, a1 = 0.0f;
  if constexpr (LOWP) {
    const float m = vmax(m_sl[0], m_sl[NSL - 1]);
    a0 = fast_exp2((m_sl[0] - m) * c);
    a1 = fast_exp2((m_sl[NSL - 1] - m) * c);
    swap32(l_sl[0] * a0 + l_sl[NSL - 1] * a1, la, lb);
  } else {
    swap32(l_sl[0], la, lb);
  }
  const float inv = LOWP ? DTy::round(1.0f / (la + lb)) : 1.0f / (la + lb);
  if constexpr (LOWP) {
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o_acc[db][r] = DTy::round(o_acc[db][r] * a0 + o_sl[NSL - 1][db][r] * a1);
    }
  }
  uint16_t* orow = op + (int64_t)my_q * p.o_ss;
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      const uint32_t x0a = DTy::pack(o_acc[db][4 * g] * inv, o_acc[db][4 * g + 1] * inv);
      const uint32_t x1a = DTy::pack(o_acc[db][4 * g + 2] * inv, o_acc[db][4 * g + 3] * inv);
      const uint32_t x0b = DTy::pack(o_acc[db][4 * g + 4] * inv, o_acc[db][4 * g + 5] * inv);
      const uint32_t x1b = DTy::pack(o_acc[db][4 * g + 6] * inv, o_acc[db][4 * g + 7] * inv);
      const auto x0 = __builtin_amdgcn_permlane32_swap(x0a, x0b, false, false);
      const auto x1 = __builtin_amdgcn_permlane32_swap(x1a, x1b, false, false);
      const int d = 32 * db + 8 * (g + hl);
      if ((!TAIL || my_q < S) && d < d_real)
        *(u32x4*)(orow + d) = u32x4{(uint32_t)x0[0], (uint32_t)x1[0], (uint32_t)x0[1], (uint32_t)x1[1]};
    }
  }
}

}  // namespace ta

// ta_fwd_rows_<dtype>_d<D>_c<causal>_t<tail>: 256 threads, B * H * ceil(S / 128) workgroups.
// The t0 variants need S to be a multiple of 128.
#define TA_ROWS_DEFINE(DTN, DT, D, C, T, WPS)                                               \
  extern "C" __global__ void __launch_bounds__(64 * ta::kRowsWaves)                         \
      __attribute__((amdgpu_waves_per_eu(WPS, WPS)))                                        \
      ta_fwd_rows_##DTN##_d##D##_c##C##_t##T(ta::FwdParams p) {                             \
    ta::attn_fwd_rows_body<DT, D, (C != 0), (T != 0)>(p);                                   \
  }
#define TA_ROWS_DEFINE_CT(DTN, DT, D, WPS)   \
  TA_ROWS_DEFINE(DTN, DT, D, 0, 0, WPS)      \
  TA_ROWS_DEFINE(DTN, DT, D, 0, 1, WPS)      \
  TA_ROWS_DEFINE(DTN, DT, D, 1, 0, WPS)      \
  TA_ROWS_DEFINE(DTN, DT, D, 1, 1, WPS)

// Input-dtype accumulation, tiles (128, TN): ta_fwd_rowsl_n<TN>_<dtype>_d<D>_c<causal>_t<tail>.
#define TA_ROWSL_DEFINE(TN, DTN, DT, D, C, T, WPS)                                          \
  extern "C" __global__ void __launch_bounds__(64 * ta::kRowsWaves)                         \
      __attribute__((amdgpu_waves_per_eu(WPS, WPS)))                                        \
      ta_fwd_rowsl_n##TN##_##DTN##_d##D##_c##C##_t##T(ta::FwdParams p) {                    \
    ta::attn_fwd_rows_body<DT, D, (C != 0), (T != 0), TN>(p);                               \
  }
#define TA_ROWSL_DEFINE_CT(TN, DTN, DT, D, WPS)   \
  TA_ROWSL_DEFINE(TN, DTN, DT, D, 0, 0, WPS)      \
  TA_ROWSL_DEFINE(TN, DTN, DT, D, 0, 1, WPS)      \
  TA_ROWSL_DEFINE(TN, DTN, DT, D, 1, 0, WPS)      \
  TA_ROWSL_DEFINE(TN, DTN, DT, D, 1, 1, WPS)
