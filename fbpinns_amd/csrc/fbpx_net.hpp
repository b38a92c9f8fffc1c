// Forward and backward jet kernels over (point, subdomain) pairs.
//
// Work decomposition: one workgroup (4 waves) per bin, a bin being a run of
// chunks (a chunk = a run of pairs of a single subdomain) processed in order;
// each wave processes 16 pairs at a time ("sub-tile").
// Lane l handles pair (l & 15) of the sub-tile and hidden units
//   u = 16*rb + 4*(l >> 4) + r,   rb < H/16, r < 4,
// which is exactly the row set that lane holds in the D layout of the 16x16
// matrix instructions (D[i][j]: lane = j + 16*(i/4), reg = i%4).  Because the
// contraction index of an MFMA may be permuted freely, a K-step of 32 takes
// the B operand's eight values of lane group g from registers [2q][0..3] and
// [2q + 1][0..3] (units 32q + 16b + 4g + ks) and the A operand with the
// matching weight columns, so a layer's output registers are directly the
// next layer's input registers.
//
// Hidden-layer products run on the f16 matrix cores at float32 accuracy: each
// float32 operand is carried as x = hi + lo with hi = f16(x), lo = f16(x - hi)
// (22 bits and the sign of the rest), and a product is hi hi + hi lo + lo hi
// with float32 accumulation.  v_mfma_f32_16x16x32_f16 does 32 contraction
// steps in the time the float32 instruction does two, so the three products
// cost 3/16 of the float32 matrix time, and they leave the vector ALU free
// (a float32 MFMA does not overlap it).  Measured on [16 x 64] x [64 x 16]
// products of uniform weights and tanh values against float64: relative
// 2-norm error 8.7e-8, against 1.44e-7 for the float32 instruction's chain of
// fused multiply-adds.  f16 has a narrow exponent range, so everything that is
// not bounded by 1 is scaled by powers of two chosen per chunk (Scales):
// weights by their largest value, tangents by theirs, gradients by a bound
// formed from the chunk's upstream gradients; the inverse factors are exact
// and ride on per-pair scalars.  Small operands keep an absolute error: 2^-39 of
// the subdomain's largest weight (16 units: 2^-50), 2^-27 of the axis' largest
// tangent, 2^-40 of the gradients' bound.
//
// Reference math (per pair, trainers.py:113-118 with the tangents that the
// nested jvp of trainers.py:213-247 pushes through):
//   xh = (x - mu)/sd, tangent e_i/sd_i          decompositions.py:184-188
//   z = W a + b, a = tanh(z) with jets
//     a0 = h, a_i = d1 z_i, a_ii = d1 z_ii + d2 z_i^2 (d1 = 1-h^2, d2 = -2 h d1)
//   u = (WL a + bL) * sd_u + mu_u               networks.py:60-68, 200-201
//   uw = u * w (Leibniz), w = cosine window     windows.py:25-35
//
// Layer-1 jets are never stored: with h, d1, d2 of layer 1 and
// zt_i = W1[:, i] / sd_i (per subdomain), a1_0 = h, a1_i = d1 zt_i and
// a1_ii = d2 zt_i^2, so the B operand of every layer-2 MFMA is rebuilt from h
// with one or two multiplies.  Layer 2 is evaluated one axis at a time (Z_0,
// then Z_i per axis).
#pragma once

#include "fbpx_common.hpp"

namespace fbpx {

// LDS copy of a subdomain's parameters except W2 (which is staged separately
// in the padded layouts below): W1 [u][i], B1, B2 (NH == 2), WL, BL.
template <int XD, int H, int NH>
struct Small {
  static constexpr int W1 = 0;
  static constexpr int B1 = H * XD;
  static constexpr int B2 = B1 + H;
  static constexpr int WL = B2 + (NH == 2 ? H : 0);
  static constexpr int BL = WL + H;
  static constexpr int N = BL + 1;
};

// Pair indices are unsigned: loads run up to 1,024 pairs ahead of the chunk's
// end before they are compared with it, which passes int32 for lists near its
// end.

// The threads that run one chunk: the workgroup, or with WAVE one wave (a
// workgroup's four waves then run four chunks of their own).  A wave's LDS
// operations are performed in order, so a wavefront-scope fence orders its
// writes before its reads where the workgroup needs a barrier.
template <bool WAVE>
struct Team {
  __device__ static int tid() { return WAVE ? (int)(threadIdx.x & 63) : (int)threadIdx.x; }
  __device__ static int size() { return WAVE ? 64 : (int)blockDim.x; }
  __device__ static int wave() { return WAVE ? 0 : (int)(threadIdx.x >> 6); }   // within the team
  __device__ static int nw() { return WAVE ? 1 : (int)(blockDim.x >> 6); }
  __device__ static int index() { return WAVE ? (int)(threadIdx.x >> 6) : 0; }  // team of the workgroup
  __device__ static void sync() {
    if constexpr (WAVE)
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    else
      __syncthreads();
  }
};

// The network's small parameters to LDS in two halves, so that a chunk's other
// first loads can be issued between them: load() issues every global load of
// the team's share (registers), store() writes them to LDS.  Teams of 64 or
// more threads (IT covers a 64-thread team; wider teams leave later slots
// unused).
template <int XD, int H, int NH, bool WAVE = false>
struct SmallStage {
  using L = Layout<XD, H, NH>;
  using SM = Small<XD, H, NH>;
  static constexpr int IT = (SM::N + 63) / 64;
  float r[IT];
  __device__ void load(const float* th) {
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = Team<WAVE>::tid() + j * Team<WAVE>::size();
      if (i < SM::N) r[j] = th[i < SM::B2 ? i : (i < SM::WL ? L::B2 + (i - SM::B2) : L::WL + (i - SM::WL))];
    }
  }
  __device__ void store(float* ss) const {
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = Team<WAVE>::tid() + j * Team<WAVE>::size();
      if (i < SM::N) ss[i] = r[j];
    }
  }
};

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// x0, x1 -> packed (hi, hi) and (lo, lo), x = hi + lo (both rounded to
// nearest).  one: 1.f in a scalar register the optimiser cannot see through,
// so that x - hi is one v_fma_mix_f32 on the packed half; the empty asm keeps
// the packed conversion from being redone per element.
__device__ inline void split2(float x0, float x1, float one, uint32_t& hi, uint32_t& lo) {
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2v{x0, x1}, h2v));
  asm("" : "+v"(hi));
  const h2v h = __builtin_bit_cast(h2v, hi);
  const f2v r = {fmaf(x0, one, -(float)h[0]), fmaf(x1, one, -(float)h[1])};
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, h2v));
}

__device__ inline float opaque_one() {
  float one = 1.f;
  asm("" : "+s"(one));
  return one;
}

// A lane's H/16 x 4 values of one pair as two f16 halves: hi[2 rb + c] packs
// units 16 rb + 4 g + 2c and + 2c + 1.  b(q): the B operand of K-step q
// (H >= 32: blocks 2q and 2q + 1; H = 16: one block, hi twice).
template <int H>
struct Split {
  static constexpr int NRB = H / 16;
  uint32_t hi[2 * NRB], lo[2 * NRB];
  template <class V>
  __device__ void set(const V& v, float one) {
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
      for (int c = 0; c < 2; ++c) split2(v[rb][2 * c], v[rb][2 * c + 1], one, hi[2 * rb + c], lo[2 * rb + c]);
  }
  __device__ h8v b(const uint32_t* p, int q) const {
    return __builtin_bit_cast(h8v, u4v{p[(4 * q) % (2 * NRB)], p[(4 * q + 1) % (2 * NRB)],
                                       p[(4 * q + 2) % (2 * NRB)], p[(4 * q + 3) % (2 * NRB)]});
  }
};

__device__ inline f4 mfma_k32(h8v a, h8v b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// 2^e with m 2^e <= 2^top (within a factor of two below it), e within
// [-126, lim]: every finite m is reached (top >= 2), and so are finite values
// under a bound m that overflowed to infinity; the clamps keep the factor and
// its inverse finite.
__device__ inline float pow2_scale(float m, int top, int lim) {
  int e = top + 126 - (int)((__builtin_bit_cast(uint32_t, m) >> 23) & 255u);
  e = e < -126 ? -126 : (e > lim ? lim : e);
  return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
}
__device__ inline float pow2_inv(float s) {   // 1 / s for s = 2^e, |e| < 127
  return __builtin_bit_cast(float, (uint32_t)(254u << 23) - __builtin_bit_cast(uint32_t, s));
}
// the same value in every lane, as a scalar
__device__ inline float uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// A chunk's box: its window constants and 1 / sd, wave-uniform values that
// every tile reads, in scalar registers (as results of vector arithmetic they
// would hold four or five vector registers per axis across the tile loop).
template <int XD>
struct ChunkBox : WindowBox<XD> {
  float isd[XD];
  __device__ inline explicit ChunkBox(const Dom& d) : WindowBox<XD>(d) {
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      isd[i] = uniform(1.f / ((d.xmax[i] - d.xmin[i]) / 2.f));
      this->mu[i] = uniform(this->mu[i]);
      this->hk[i] = uniform(this->hk[i]);
      this->n2k[i] = uniform(this->n2k[i]);
      this->kk[i] = uniform(this->kk[i]);
    }
  }
};

// Powers of two of one chunk (all exact):
//   W2 2^w and (diag(WL) W2) 2^r are at most 2^14 in LDS,
//   zt_i 2^e[i] is at most 4 (table ztS),
//   the upstream gradients are carried times 2^k (backward).
template <int XD>
struct Scales {
  float w, iw, r, ir, e[XD], ie[XD], k, ik;
};

// Lane-major LDS fragments of W2 (f16 hi / lo): the MFMA A operands of one
// K-step q and 16-row block ob for all 64 lanes.  With lane l = 16g + pl,
// H >= 32: fragment f = (q NRB + ob) 2 + piece holds 8 halves per lane,
//   wt: W2[16ob + pl][k] 2^w, k = 32q + 16b + 4g + ks at 4b + ks
//   wr: (WL_k W2[k][16ob + pl]) 2^r, same k         (A of (diag(WL) W2)^T . g)
// H = 16: a fragment of 4 hi then 4 lo halves per lane (k = 4g + ks) and one of
// the 4 rests x - hi - lo and 4 zeros, which carries the weights whole.  (A
// weight's rounding to 22 bits is the same for every pair and does not average
// out over them; with 16 terms per unit it shows: first bias gradients of Burgers
// at 7 % more error than with float32 products, 0 % with the rests.  At h = 32 and
// 64 it is below 2 %.  One more matrix instruction and LDS read per product:
// forward of 162,000 pairs of [2,16,16,1] networks 18.9 -> 19.6 us.)
// Consecutive lanes read consecutive 16-byte slots: conflict-free.
// The weights come from memory once, coalesced, through a padded f32 copy in
// LDS (which may lie where the fragments go: they are written after the
// barrier that follows the last read).  Gathered from memory in fragment
// order, the staging of a chunk took 34,000 cycles at H = 64 and 17,700 at
// H = 32.
template <int H>
struct W2Frags {
  static constexpr int NRB = H / 16;
  static constexpr int NQ = H >= 32 ? H / 32 : 1;
  static constexpr int NEL = H >= 32 ? 8 : 4;         // weights per item
  static constexpr int ITEMS = NQ * NRB * 64;
  static constexpr int IT = (ITEMS + 255) / 256;      // items per thread of a 256-thread workgroup
  static constexpr int LDW = H + 4;                   // row of the f32 copy: 16 rows start in 16 bank groups
  static constexpr int TMP = H * LDW;
  static constexpr int SET = H >= 32 ? H * H : 2 * H * H;   // floats of a fragment set
  static constexpr int RAW = H * H / 256;
  float raw[RAW], a[IT][NEL], c[IT][NEL];
  __device__ static int unit(int q, int g, int j) { return 32 * q + 16 * (j >> 2) + 4 * g + (j & 3); }
  __device__ void load(const float* w2) {
#pragma unroll
    for (int j = 0; j < RAW; ++j) raw[j] = w2[(int)threadIdx.x + 256 * j];
  }
  __device__ void stash(float* tmp) const {
#pragma unroll
    for (int j = 0; j < RAW; ++j) {
      const int i = (int)threadIdx.x + 256 * j;
      tmp[(i / H) * LDW + i % H] = raw[j];
    }
  }
  template <bool WR>
  __device__ void read(const float* tmp, const float* wl) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = (int)threadIdx.x + 256 * it, l = t & 63, g = l >> 4, pl = l & 15, f = t >> 6;
      const int q = f / NRB, ob = f % NRB;
      if (t >= ITEMS) continue;
#pragma unroll
      for (int b = 0; b < NEL / 4; ++b) {
        const f4 v = *reinterpret_cast<const f4*>(tmp + (16 * ob + pl) * LDW + unit(q, g, 4 * b));
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) a[it][4 * b + ks] = v[ks];
      }
      if (WR) {
#pragma unroll
        for (int j = 0; j < NEL; ++j) {
          const int k = unit(q, g, j);
          c[it][j] = tmp[k * LDW + 16 * ob + pl] * wl[k];
        }
      }
    }
  }
  // this thread's largest |value|.  (An infinite or NaN weight makes its
  // subdomain's values NaN: hi + lo of an infinity is inf - inf.)
  __device__ static float largest(const float (*v)[NEL]) {
    float m = 0.f;
#pragma unroll
    for (int it = 0; it < IT; ++it)
      if ((int)threadIdx.x + 256 * it < ITEMS) {
#pragma unroll
        for (int j = 0; j < NEL; ++j) m = fmaxf(m, fabsf(v[it][j]));
      }
    return m;
  }
  __device__ static void store(const float (*v)[NEL], float scale, float one, float* dst) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = (int)threadIdx.x + 256 * it, l = t & 63, f = t >> 6;
      if (t >= ITEMS) continue;
      uint32_t hi[NEL / 2], lo[NEL / 2];
#pragma unroll
      for (int c = 0; c < NEL / 2; ++c) split2(v[it][2 * c] * scale, v[it][2 * c + 1] * scale, one, hi[c], lo[c]);
      uint32_t* w = reinterpret_cast<uint32_t*>(dst);
      if constexpr (H >= 32) {
        *reinterpret_cast<u4v*>(w + (2 * f * 64 + l) * 4) = u4v{hi[0], hi[1], hi[2], hi[3]};
        *reinterpret_cast<u4v*>(w + ((2 * f + 1) * 64 + l) * 4) = u4v{lo[0], lo[1], lo[2], lo[3]};
      } else {
        uint32_t rest[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const h2v h = __builtin_bit_cast(h2v, hi[c]), m = __builtin_bit_cast(h2v, lo[c]);
          const f2v r = {(v[it][2 * c] * scale - (float)h[0]) - (float)m[0],
                         (v[it][2 * c + 1] * scale - (float)h[1]) - (float)m[1]};
          rest[c] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, h2v));
        }
        *reinterpret_cast<u4v*>(w + l * 4) = u4v{hi[0], hi[1], lo[0], lo[1]};
        *reinterpret_cast<u4v*>(w + 256 + l * 4) = u4v{rest[0], rest[1], 0u, 0u};
      }
    }
  }
};

// Sum over the four 16-lane rows (lane groups g) for every pl, in registers:
// v_permlane32_swap exchanges the upper half of its first operand with the
// lower half of its second, so with both holding v the two results add to
// v[l] + v[l ^ 32]; v_permlane16_swap does the same between odd and even
// rows.  Written as asm: the compiler builtins for these instructions read
// one result register twice on this toolchain.  The s_nop covers the
// VALU-write -> permlane-read hazard.
__device__ inline float sum_groups(float v) {
  float a = v, b = v;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  float s = a + b;
  a = s;
  b = s;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return a + b;
}

template <int CTRL>
__device__ inline float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// One stage of a reduce-scatter of maxima over a DPP row (see split_stage).
template <int N, int CTRL>
__device__ inline void max_stage(float* v, bool upper) {
#pragma unroll
  for (int k = 0; k < N / 2; ++k) {
    const float lo = v[k], hi = v[k + N / 2];
    v[k] = fmaxf(upper ? hi : lo, dpp<CTRL>(upper ? lo : hi));
  }
}

// Lane pl of every row gets the largest v[pl] over the wave (v >= 0), the 16
// values together: 60 instructions, where a butterfly per value took 45 each.
__device__ inline float max_wave16(float* v, int pl) {
  max_stage<16, 0x140>(v, (pl >> 3) & 1);
  max_stage<8, 0x141>(v, (pl >> 2) & 1);
  max_stage<4, 0x1B>(v, (pl >> 1) & 1);
  max_stage<2, 0xB1>(v, pl & 1);
  float a = v[0], b = v[0];
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  a = b = fmaxf(a, b);
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

// Sum of v over the 16 lanes of a row, in every lane of it.
__device__ inline float sum_row(float v) {
  v += dpp<0x140>(v);
  v += dpp<0x141>(v);
  v += dpp<0x1B>(v);
  return v + dpp<0xB1>(v);
}

// One reduce-scatter stage over a DPP row: lanes whose stage bit is set keep
// the upper half of v[0..N), the others the lower half; each adds the half
// its partner (DPP control CTRL, a lane with the opposite bit) does not keep.
template <int N, int CTRL>
__device__ inline void split_stage(float* v, bool upper) {
#pragma unroll
  for (int k = 0; k < N / 2; ++k) {
    const float lo = v[k], hi = v[k + N / 2];
    const float send = upper ? lo : hi;
    const float keep = upper ? hi : lo;
    v[k] = keep + dpp<CTRL>(send);
  }
}

// The two mirror stages with whole DPP banks (4 lanes) on each side: lanes
// of the banks in the low mask keep lo + partner's lo, the others hi +
// partner's hi, written by two bank-masked DPP adds into one register (no
// selects).  row_mirror pairs pl with 15 - pl (banks 0,1 | 2,3),
// row_half_mirror pl with pl ^ 7 (banks 0,2 | 1,3).  One asm block per
// stage; its leading s_nop covers the VALU-write -> DPP-read hazard on the
// operands (the later pairs' operands are older still).
#define FBPX_DPP_PAIR(CTRL, LO, HI, D, A, B)                               \
  "v_add_f32_dpp %" #D ", %" #A ", %" #A " " CTRL " row_mask:0xf bank_mask:" LO "\n\t" \
  "v_add_f32_dpp %" #D ", %" #B ", %" #B " " CTRL " row_mask:0xf bank_mask:" HI "\n\t"

__device__ inline void mirror_stage(float* v) {
  float d[8];
  asm("s_nop 1\n\t"
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 0, 8, 16)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 1, 9, 17)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 2, 10, 18)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 3, 11, 19)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 4, 12, 20)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 5, 13, 21)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 6, 14, 22)
      FBPX_DPP_PAIR("row_mirror", "0x3", "0xc", 7, 15, 23)
      : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3]), "=&v"(d[4]), "=&v"(d[5]), "=&v"(d[6]), "=&v"(d[7])
      : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]),
        "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]), "v"(v[12]), "v"(v[13]), "v"(v[14]), "v"(v[15]));
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = d[k];
}

__device__ inline void half_mirror_stage(float* v) {
  float d[4];
  asm("s_nop 1\n\t"
      FBPX_DPP_PAIR("row_half_mirror", "0x5", "0xa", 0, 4, 8)
      FBPX_DPP_PAIR("row_half_mirror", "0x5", "0xa", 1, 5, 9)
      FBPX_DPP_PAIR("row_half_mirror", "0x5", "0xa", 2, 6, 10)
      FBPX_DPP_PAIR("row_half_mirror", "0x5", "0xa", 3, 7, 11)
      : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3])
      : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = d[k];
}
#undef FBPX_DPP_PAIR

// vals[rb][r] holds this lane's contribution for unit 16rb + 4g + r.  Sums
// every entry over the 16 pair-lanes of the row and returns the total for
// unit 16*(pl/4) + 4g + pl%4 to lane pl < 4 NRB (lane pl owns that unit; no
// two lanes of a wave own the same).  Butterfly reduce-scatter: partners
// row_mirror (pl ^ 15), row_half_mirror (pl ^ 7), quad_perm[3,2,1,0]
// (pl ^ 3), quad_perm[1,0,3,2] (pl ^ 1) flip bits 3, 2, 1, 0 of pl in turn
// while sharing the bits above; with fewer than 16 values the top stages
// are plain additions.  After the last stage lane pl holds the total of
// value index pl & (V - 1).
template <int NRB>
__device__ inline float reduce_units(const float (*vals)[4], int pl) {
  constexpr int V = NRB * 4;
  float v[V];
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) v[4 * rb + r] = vals[rb][r];
  if constexpr (V <= 8) {
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] += dpp<0x140>(v[k]);
  }
  if constexpr (V <= 4) {
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] += dpp<0x141>(v[k]);
  }
  if constexpr (V == 16) mirror_stage(v);
  if constexpr (V >= 8) half_mirror_stage(v);
  split_stage<4, 0x1B>(v, (pl >> 1) & 1);
  split_stage<2, 0xB1>(v, pl & 1);
  return v[0];
}

// dst[kind * h + the lane's unit of reduce_units] = v[kind]
template <int NRB, int NK>
__device__ inline void store_units(float* dst, const float* v, int h, int pl, int g) {
#pragma unroll
  for (int j = 0; j < NK; ++j)
    if (pl < 4 * NRB) dst[j * h + 16 * (pl >> 2) + 4 * g + (pl & 3)] = v[j];
}

// Hide the values of a register tile from the optimiser (an empty asm that
// "may modify" each element), so that quantities derived from them (tanh
// derivatives) are recomputed where used instead of being kept alive across
// the axis phases, which would cost 16 registers per derived tile.
template <int NRB>
__device__ inline void opaque(float (*a)[4]) {
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(a[rb][r]));
}

// v[c] for a wave-uniform runtime index c < N (selects, no register indexing).
template <int N>
__device__ inline float pick(const float* v, int c) {
  float r = v[0];
#pragma unroll
  for (int k = 1; k < N; ++k) r = (c == k) ? v[k] : r;
  return r;
}

// tanh derivatives from h = tanh(z): d1 = 1 - h^2, d2 = -2 h d1, d3 = -2 (d1^2 + h d2)
__device__ inline float tanh_d1(float h) { return 1.f - h * h; }
__device__ inline float tanh_d2(float h) { return -2.f * h * (1.f - h * h); }
__device__ inline float tanh_d3(float h) {
  const float d1 = 1.f - h * h;
  return -2.f * (d1 * d1 - 2.f * h * h * d1);
}

// Per-subdomain layer-1 tangent tables in LDS: with zt_i[u] = W1[u][i] / sd_i,
//   zt[i*H + u] = zt_i[u],  zt[XD*H + i*H + u] = -2 zt_i[u]^2;
// a third table zt_i[u] 2^e[i] follows them with two hidden layers (stage_two).
template <int XD, int H, class SM, bool WAVE = false>
__device__ inline void stage_zt(const float* ss, const float* isd, float* zt) {
  for (int t = Team<WAVE>::tid(); t < XD * H; t += Team<WAVE>::size()) {
    const int i = t / H, u = t % H;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < XD; ++j) {
      // opaque: selects between the values, not between their addresses
      // (which would put the array in memory)
      float sj = isd[j];
      asm("" : "+v"(sj));
      s = i == j ? sj : s;
    }
    const float z = ss[SM::W1 + u * XD + i] * s;
    zt[t] = z;
    zt[XD * H + t] = -2.f * z * z;
  }
}

// Per-lane LDS base pointers (lane group g = lane >> 4, pl = lane & 15).
// Every LDS read in the pair loops is one of these plus a compile-time
// offset, so an array costs one address register (ds_read immediate
// offsets) rather than one per access pattern.
//   w1  = ss + W1 + 4g*XD      W1[16rb + 4g + r][i]        at [(16rb + r)*XD + i]
//   vec = ss + 4g              B1/B2/WL[16rb + 4g + r]     at [off + 16rb + r]
//   zt  = szt + 4g             zt[i][16rb + 4g + r]        at [i*H + 16rb + r]
//   z2, zs: the -2 zt^2 and zt 2^e tables, same indexing
//   wt  = swt + lane*4         fragment f of W2 (W2Frags) at [f*256]
//   wr  = swr + lane*4         fragment f of the transposed set, same
struct LaneLds {
  const float* w1;
  const float* vec;
  const float* zt;
  const float* z2;
  const float* zs;
  const float* wt;
  const float* wr;
};

template <int XD, int H, class SM>
__device__ inline LaneLds lane_lds(const float* ss, const float* szt, const float* swt, const float* swr, int pl,
                                   int g) {
  LaneLds v;
  v.w1 = ss + SM::W1 + 4 * g * XD;
  v.vec = ss + 4 * g;
  v.zt = szt + 4 * g;
  v.z2 = szt + XD * H + 4 * g;
  v.zs = szt + 2 * XD * H + 4 * g;
  v.wt = swt + (16 * g + pl) * 4;
  v.wr = swr + (16 * g + pl) * 4;
  return v;
}

// The fragments of one 16-row block (all K-steps).  A pass takes its first
// block's as an argument, so that the caller can issue those reads before the
// vector work that forms the B operand: read inside the pass, every pass
// began with an LDS round trip that the other wave of the SIMD did not cover.
template <int H>
struct FragRow {
  static constexpr int NQ = W2Frags<H>::NQ;
  h8v hi[NQ], lo[NQ];   // H = 16: hi[0] = 4 hi and 4 lo weights, lo[0] = their rests
  __device__ void load(const float* frag, int ob) {
    if constexpr (H >= 32) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        hi[q] = *reinterpret_cast<const h8v*>(frag + (q * (H / 16) + ob) * 512);
        lo[q] = *reinterpret_cast<const h8v*>(frag + (q * (H / 16) + ob) * 512 + 256);
      }
    } else {
      hi[0] = *reinterpret_cast<const h8v*>(frag);
      lo[0] = *reinterpret_cast<const h8v*>(frag + 256);
    }
  }
};

// Block 0 of a fragment set, its reads pinned here.
template <int H>
__device__ inline FragRow<H> frag_head(const float* frag) {
  FragRow<H> f;
  f.load(frag, 0);
  __builtin_amdgcn_sched_barrier(0);
  return f;
}

// Z[ob] += fragments (LDS, see W2Frags) times the split B operand.  The two
// small products of every K-step are accumulated before the large ones, whose
// rounding then happens once per K-step: 8.7e-8 relative error at H = 64
// where one K-step after the other gives about 1e-7.
template <int H>
__device__ inline void frag_pass(const float* frag, FragRow<H> f, const Split<H>& b, f4* Z) {
  using F = W2Frags<H>;
  constexpr int NRB = H / 16;
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (H >= 32) {
#pragma unroll
    for (int ob = 0; ob < NRB; ++ob) {
      FragRow<H> n;
      if (ob + 1 < NRB) n.load(frag, ob + 1);
#pragma unroll
      for (int q = 0; q < F::NQ; ++q) {
        Z[ob] = mfma_k32(f.lo[q], b.b(b.hi, q), Z[ob]);
        Z[ob] = mfma_k32(f.hi[q], b.b(b.lo, q), Z[ob]);
      }
#pragma unroll
      for (int q = 0; q < F::NQ; ++q) Z[ob] = mfma_k32(f.hi[q], b.b(b.hi, q), Z[ob]);
      if (ob + 1 < NRB) f = n;
    }
    // the reads of the next row block go between this block's MFMAs
    constexpr int NR = 2 * F::NQ, NM = 3 * F::NQ;
#pragma unroll
    for (int ob = 0; ob + 1 < NRB; ++ob) {
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NM - NR, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
  } else {
    // one K-step of 16: the rests against hi, then hi and lo weights side by
    // side in a K of 32 against lo twice (which adds the lo lo product) and hi
    // twice
    Z[0] = mfma_k32(f.lo[0], b.b(b.hi, 0), Z[0]);
    Z[0] = mfma_k32(f.hi[0], b.b(b.lo, 0), Z[0]);
    Z[0] = mfma_k32(f.hi[0], b.b(b.hi, 0), Z[0]);
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int H>
__device__ inline void frag_mul(const float* frag, const FragRow<H>& head, const Split<H>& b, f4* Z) {
#pragma unroll
  for (int ob = 0; ob < H / 16; ++ob) Z[ob] = f4{0.f, 0.f, 0.f, 0.f};
  frag_pass<H>(frag, head, b, Z);
}

// Layer 1 for this lane's units (rows 16rb + 4g + r): h = tanh(W1 xh + b1).
template <int XD, int H, class SM>
__device__ inline void layer1_stream(const LaneLds& v, const float* xh, float (*h1)[4]) {
#pragma unroll
  for (int rb = 0; rb < H / 16; ++rb) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float z = v.vec[SM::B1 + 16 * rb + r];
#pragma unroll
      for (int i = 0; i < XD; ++i) z = fmaf(v.w1[(16 * rb + r) * XD + i], xh[i], z);
      h1[rb][r] = tanh_f(z);
    }
  }
}

// Z_0 2^w = (W2 h1 + b2) 2^w (b2 is staged times 2^w).
template <int H, class SM>
__device__ inline void layer2_value(const LaneLds& v, const float (*h1)[4], float one, f4* Z) {
#pragma unroll
  for (int ob = 0; ob < H / 16; ++ob) {
    const float* b2 = v.vec + SM::B2 + 16 * ob;
    Z[ob] = f4{b2[0], b2[1], b2[2], b2[3]};
  }
  const FragRow<H> head = frag_head<H>(v.wt);
  Split<H> b;
  b.set(h1, one);
  frag_pass<H>(v.wt, head, b, Z);
}

// a[rb][r] zs[zrow + ...]: the B operand e1 zt_i 2^e[i] of axis i (zrow = i H).
template <int H>
__device__ inline void tangent_split(const LaneLds& v, const float (*e1)[4], int zrow, float one, Split<H>& b) {
  float t[H / 16][4];
#pragma unroll
  for (int rb = 0; rb < H / 16; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) t[rb][r] = e1[rb][r] * v.zs[zrow + 16 * rb + r];
  b.set(t, one);
}

// The pair's layer-1 combination of every tangent the upstream gradient
// asks for, s = sum_i (gur_i a1_i + gur_ii a1_ii) with a1_i = e1 zt_i and
// a1_ii = e2 zt_i^2 (e1 = 1 - h1^2, e2 = -2 h1 e1, e3 = e1 (4 - 6 e1)):
//   s = e1 (A + h1 B),  A = sum_i gur_i zt_i,  B = sum_i gur_ii (-2 zt_i^2),
// and -1 / (2 e1) times the factor that the W2^T vector vt multiplies in the
// layer-1 gradient,
//   e2 A + e3 sum_i gur_ii zt_i^2 = -2 e1 rv,  rv = h1 A + (1 - 1.5 e1) B.
template <class S, int H>
__device__ inline void pair_s(const LaneLds& v, const float (*h1)[4], const float* gur, float (*sv)[4],
                              float (*rv)[4]) {
#pragma unroll
  for (int rb = 0; rb < H / 16; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float A = 0.f, B = 0.f;
      bool a = false, b = false;
#pragma unroll
      for (int i = 0; i < S::XD; ++i) {
        if (S::has1(i)) {
          const float t = v.zt[i * H + 16 * rb + r], g = gur[S::col1(i)];
          A = a ? fmaf(g, t, A) : g * t;
          a = true;
        }
        if (S::has2(i)) {
          const float t = v.z2[i * H + 16 * rb + r], g = gur[S::col2(i)];
          B = b ? fmaf(g, t, B) : g * t;
          b = true;
        }
      }
      const float h = h1[rb][r];
      const float e1 = fmaf(-h, h, 1.f);
      sv[rb][r] = e1 * (b ? fmaf(h, B, A) : A);
      rv[rb][r] = b ? fmaf(h, A, fmaf(-1.5f, e1, 1.f) * B) : h * A;
    }
}

// Stages one subdomain of a two-hidden-layer network in LDS: the small
// parameters, the tangent tables and the f16 fragments of W2 (and with WR of
// diag(WL) W2), and forms the chunk's scales.  With BWD, grad_max() (called
// once the weights' loads are issued) returns this thread's largest |upstream
// gradient| per jet column over its share of the chunk's pairs, and the gradients' scale k is chosen from a bound on every
// gradient value that enters a product: with R the largest absolute row sum
// of W2, ZB_i = max_o sum_u |W2[o][u] zt_i[u]| >= |Z_i|, ZT_i = max |zt_i| and
// g the bound on gur (window jets |w| <= 1, |w_i| <= 0.65 k_i, |w_ii| <= k_i^2
// with k_i = pi / sd_i; |2 h e1|, |f2| <= 0.77, |f3| <= 2):
//   |s| <= bS = sum_i g_i ZT_i + 0.77 g_ii ZT_i^2,
//   |G_i| 2^-e[i] <= 0.77 g_ii ZB_i ZT_i,  |G_0| <= g_0 + 0.77 R bS + 2 sum_i g_ii ZB_i^2.
// Typical values lie 2^-8 to 2^-12 below the bound; the f16 pairs hold 22
// bits down to 2^-17 below it and 2^-40 of the bound absolutely after that.
// All threads of the workgroup; ends with a barrier.
template <class S, int H, class SM, bool WR, bool BWD, class GradMax>
__device__ inline void stage_two(const float* th, const Dom& d, const float* isd, GradMax grad_max, float one,
                                 float* ss, float* szt, float* swt, float* swr, float* red, Scales<S::XD>& sc) {
  constexpr int XD = S::XD, J = S::J;
  using L = Layout<XD, H, 2>;
  using F = W2Frags<H>;
  constexpr int RW = 0, RR = 1, RT = 2, RS = RT + XD, RZ = RS + 1, RG = RZ + XD, NR = BWD ? RG + J : RS;
  static_assert(NR <= 16, "one row of lanes reduces them all");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  F f;
  SmallStage<XD, H, 2> st;
  st.load(th);
  f.load(th + L::W2);
  const float* gm = grad_max();
  st.store(ss);
  f.stash(swt);
  __syncthreads();
  stage_zt<XD, H, SM>(ss, isd, szt);
  f.template read<WR>(swt, ss + SM::WL);
  __syncthreads();
  float m[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) m[i] = 0.f;
#pragma unroll
  for (int i = 0; i < XD; ++i) m[RT + i] = fabsf(szt[i * H + lane % H]);
  m[RW] = F::largest(f.a);
  m[RR] = WR ? F::largest(f.c) : 0.f;
  if constexpr (BWD) {
    // row sums: a wave's items are all of one 16-row block, row 16ob + pl of
    // lane pl, so adding the lane groups completes them
    float rs = 0.f, zb[XD];
#pragma unroll
    for (int i = 0; i < XD; ++i) zb[i] = 0.f;
#pragma unroll
    for (int it = 0; it < F::IT; ++it)
      if ((int)threadIdx.x + 256 * it < F::ITEMS) {
#pragma unroll
        for (int j = 0; j < F::NEL; ++j) {
          const int k = F::unit(it, lane >> 4, j);
          const float a = fabsf(f.a[it][j]);
          rs += a;
#pragma unroll
          for (int i = 0; i < XD; ++i) zb[i] = fmaf(a, fabsf(szt[i * H + k]), zb[i]);
        }
      }
    m[RS] = sum_groups(rs);
#pragma unroll
    for (int i = 0; i < XD; ++i) m[RZ + i] = sum_groups(zb[i]);
#pragma unroll
    for (int c = 0; c < J; ++c) m[RG + c] = gm[c];
  }
  {
    const float v = max_wave16(m, lane & 15);
    if (lane < 16) red[wave * 16 + lane] = v;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NR; ++i)
    m[i] = uniform(fmaxf(fmaxf(red[i], red[16 + i]), fmaxf(red[32 + i], red[48 + i])));
  sc.w = pow2_scale(m[RW], 14, 40);
  sc.iw = pow2_inv(sc.w);
  sc.r = WR ? pow2_scale(m[RR], 14, 40) : 1.f;
  sc.ir = pow2_inv(sc.r);
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    sc.e[i] = pow2_scale(m[RT + i], 2, 40);
    sc.ie[i] = pow2_inv(sc.e[i]);
  }
  sc.k = sc.ik = 1.f;
  if constexpr (BWD) {
    const float us = fabsf(d.usd);
    float g0 = m[RG], bS = 0.f, q = 0.f, b = 0.f;
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      if (!S::has1(i)) continue;
      const float k = kPi * fabsf(isd[i]);
      const float ga = m[RG + S::col1(i)], gb = S::has2(i) ? m[RG + S::col2(i)] : 0.f;
      g0 = fmaf(0.65f * k, ga, fmaf(k * k, gb, g0));
      bS = fmaf(us * fmaf(1.3f * k, gb, ga), m[RT + i], fmaf(0.77f * us * gb, m[RT + i] * m[RT + i], bS));
      q = fmaf(2.f * us * gb, m[RZ + i] * m[RZ + i], q);
      b = fmaxf(b, 0.77f * us * gb * m[RZ + i] * m[RT + i]);
    }
    b = fmaxf(fmaxf(b, bS), fmaf(us, g0, fmaf(0.77f * m[RS], bS, q)));
    // (with the unnormalising factor in the bound, us 2^k stays below 2^100, so
    // that gradients of zero stay zero: 0 times an infinite factor is NaN)
    sc.k = uniform(pow2_scale(fmaxf(b, us * 0x1p-85f), 15, 100));
    sc.ik = pow2_inv(sc.k);
  }
  for (int t = threadIdx.x; t < XD * H; t += blockDim.x) {
    float e = sc.e[0];
#pragma unroll
    for (int j = 1; j < XD; ++j)
      if (t / H == j) e = sc.e[j];
    szt[2 * XD * H + t] = szt[t] * e;
  }
  for (int t = threadIdx.x; t < H; t += blockDim.x) ss[SM::B2 + t] *= sc.w;
  F::store(f.a, sc.w, one, swt);
  if constexpr (WR) F::store(f.c, sc.r, one, swr);
  __syncthreads();
}

// What depends on a pair alone (its window jets, normalised point, upstream
// gradient) would be formed by each of the four lane groups that share a
// 16-pair sub-tile.  The two-layer kernels form it for four sub-tiles at once,
// one pair per lane (lane group g: the g-th sub-tile), and keep it as rows of
// ROW floats in LDS, per wave; a sub-tile reads its 16 rows back (a row stride
// of 12 words: 16 four-word reads without a bank conflict).  Vector instructions
// per sub-tile, backward: 1,962 -> 1,870 (3D, h = 64), 661 -> 625 (2D, h = 32, one
// second derivative).  With the box constants in scalar registers, of 7.2 million
// pairs (3D, h = 64): backward 3,360 -> 3,210 us, forward 1,195 -> 1,160; 412,000
// pairs: 272 -> 249 and 105 -> 99.  2D, h = 32: forward 71.3 -> 69.2 us, backward 150 ->
// 148.5 (946,000 pairs), 44.3 -> 43.0 and 68 -> 63.4 (614,000).
struct PairRows {
  static constexpr int ROW = 12, WAVE = 64 * ROW;
};

// ------------------------------------------------------------------ forward

// One chunk of the forward (a run of pairs of one subdomain).
template <int XD, int H, int NH, int D1M, int D2M, bool WAVE = false>
__device__ inline void fwd_chunk(const float* __restrict__ theta, const float* __restrict__ dom,
                                 const float* __restrict__ x, const fbpx_worklist& wl, float* __restrict__ pairbuf,
                                 int chunk) {
  using S = Schema<XD, D1M, D2M>;
  using L = Layout<XD, H, NH>;
  using SM = Small<XD, H, NH>;
  using T = Team<WAVE>;
  static_assert(!WAVE || NH == 1, "one wave per chunk: one-hidden-layer networks");
  using R = PairRows;
  using F = W2Frags<H>;
  constexpr int J = S::J, NRB = H / 16, NT = WAVE ? 4 : 1;
  __shared__ float ss_[NT][SM::N];
  __shared__ float szt_[NT][(NH == 2 ? 3 : 2) * XD * H];
  // both fragment sets, or (the value alone) one, which the f32 copy outgrows
  __shared__ __attribute__((aligned(16))) float swt[NH == 2 ? (S::N1 > 0 ? 2 * F::SET : F::TMP > F::SET ? F::TMP : F::SET) : 1];
  float* const swr = swt + (NH == 2 && S::N1 > 0 ? F::SET : 0);
  __shared__ __attribute__((aligned(16))) float srow[NH == 2 ? 4 * R::WAVE : 1];
  float* const ss = ss_[T::index()];
  float* const szt = szt_[T::index()];

  const int model = wl.chunk_model[chunk];
  const uint32_t beg = wl.chunk_start[chunk], end = wl.chunk_start[chunk + 1];
  const float* th = theta + (size_t)model * L::P;
  const int lane = threadIdx.x & 63, wave = T::wave(), nw = T::nw();
  const int pl = lane & 15, g = lane >> 4;
  // the points of each sub-tile (NH == 2: of each four, PairRows) are fetched
  // one sub-tile ahead (pair index at the top of the previous sub-tile,
  // coordinates in its middle), so the two dependent global loads overlap the
  // previous sub-tile's compute; with one hidden layer the first sub-tile's
  // pair index is loaded with the parameter staging and its coordinates before
  // the staging's LDS writes and barriers (with two, the registers they would
  // hold spill others)
  float xn[XD];
  const uint32_t k0 = beg + wave * 16 + pl;
  if constexpr (NH == 1) {
    const int p0 = wl.pair_point[k0 < end ? k0 : beg];
    SmallStage<XD, H, NH, WAVE> st;
    st.load(th);
#pragma unroll
    for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)p0 * XD + i];
    st.store(ss);
  }
  Dom d;
  load_dom(dom, model, d);
  const ChunkBox<XD> box(d);
  const float* const mu = box.mu;
  const float* const isd = box.isd;
  const float one = opaque_one();
  Scales<XD> sc;
  if constexpr (NH == 1) {
    T::sync();
    stage_zt<XD, H, SM, WAVE>(ss, isd, szt);
    T::sync();
  } else {
    stage_two<S, H, SM, (S::N1 > 0), false>(th, d, isd, [] { return (const float*)nullptr; }, one, ss, szt, swt, swr,
                                            srow, sc);
  }

  const LaneLds v = lane_lds<XD, H, SM>(ss, szt, swt, swr, pl, g);
  // NH == 2: this lane's row (window jets, normalised point, slot) of the next
  // four sub-tiles
  static_assert(J + XD + 1 <= R::ROW, "a pair's row");
  float* const rows = srow + (NH == 2 ? wave * R::WAVE : 0);
  const auto put_row = [&](const float* xp, int slot) {
    float wj[J];
    window_jets<S>(xp, box, d.flag, wj);
    float* const to = rows + lane * R::ROW;
#pragma unroll
    for (int c = 0; c < J; ++c) to[c] = wj[c];
#pragma unroll
    for (int i = 0; i < XD; ++i) to[J + i] = (xp[i] - mu[i]) * isd[i];
    to[J + XD] = __int_as_float(slot);
    Team<true>::sync();
  };
  if constexpr (NH == 2) {
    const uint32_t kq = beg + wave * 16 + g * 64 + pl;
    const int pq = wl.pair_point[kq < end ? kq : beg], sq = wl.pair_slot[kq < end ? kq : beg];
#pragma unroll
    for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)pq * XD + i];
    put_row(xn, sq);
  }
  int t = 0;   // sub-tile of this wave
  for (uint32_t base = beg + wave * 16; base < end; base += nw * 16, ++t) {
    const uint32_t k = base + pl;
    const bool valid = k < end;
    const uint32_t kn = k + nw * 16;
    float xv[XD], xh[XD];
    int pn, slot;
    const float* const row = rows + (NH == 2 ? ((t & 3) * 16 + pl) * R::ROW : 0);
    const uint32_t kq = kn + g * 64;
    const bool refill = NH == 2 && (t & 3) == 3;
    int slotn;
    float xq[XD];
    if constexpr (NH == 2) {
#pragma unroll
      for (int i = 0; i < XD; ++i) xh[i] = row[J + i];
      if (refill) {
        pn = wl.pair_point[kq < end ? kq : beg];
        slotn = wl.pair_slot[kq < end ? kq : beg];
      }
    } else {
      slot = wl.pair_slot[valid ? k : beg];
      pn = wl.pair_point[kn < end ? kn : beg];
#pragma unroll
      for (int i = 0; i < XD; ++i) {
        xv[i] = xn[i];
        xh[i] = (xv[i] - mu[i]) * isd[i];
      }
    }
    float h1[NRB][4];
    layer1_stream<XD, H, SM>(v, xh, h1);
    float ur[J];
#pragma unroll
    for (int c = 0; c < J; ++c) ur[c] = 0.f;
    if constexpr (NH == 1) {
#pragma unroll
      for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)pn * XD + i];
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float wlu = v.vec[SM::WL + 16 * rb + r];
          const float h = h1[rb][r];
          ur[0] = fmaf(wlu, h, ur[0]);
#pragma unroll
          for (int i = 0; i < XD; ++i) {
            const float z = v.zt[i * H + 16 * rb + r];
            if (S::has1(i)) ur[S::col1(i)] = fmaf(wlu, tanh_d1(h) * z, ur[S::col1(i)]);
            if (S::has2(i)) ur[S::col2(i)] = fmaf(wlu, tanh_d2(h) * z * z, ur[S::col2(i)]);
          }
        }
    } else {
      f4 Z0[NRB];
      layer2_value<H, SM>(v, h1, one, Z0);
      // output-layer weights times the layer-2 tanh derivatives, per element:
      // wd1 = WL f1 and wd2 = WL f1 h2 = WL f2 / (-2), so that u_i = sum wd1 Z_i
      // and the Z_i^2 part of u_ii = sum WL (f1 Z_ii + f2 Z_i^2) costs two FMAs
      // (its factor -2 is applied to the lane's sum)
      float f1[NRB][4], wd1[NRB][4], wd2[NRB][4];
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float wlu = v.vec[SM::WL + 16 * ob + r];
          const float h = tanh_f(Z0[ob][r], sc.iw);
          ur[0] = fmaf(wlu, h, ur[0]);
          f1[ob][r] = fmaf(-h, h, 1.f);
          wd1[ob][r] = wlu * f1[ob][r];
          wd2[ob][r] = wd1[ob][r] * h;
        }
      if (refill) {
#pragma unroll
        for (int i = 0; i < XD; ++i) xq[i] = x[(size_t)pn * XD + i];
      }
      __builtin_amdgcn_sched_barrier(0);
      // sum_o WL f1 Z_c = sum_u vt[u] a1_c[u] with vt = (diag(WL) W2)^T f1: one
      // transposed pass per sub-tile replaces the Z_ii passes of every axis and
      // the Z_i passes of axes without a second derivative.  With e1 = 1 - h1^2,
      // a1_i = e1 zt_i and a1_ii = -2 h1 e1 zt_i^2, so the per-axis dot
      // products take ve = vt e1 (first order) and w = vt e1 h1 (second order).
      // Scales: vt 2^r, Z_i 2^(w + e[i]), taken off the pair's sums.
      float e1[NRB][4], ve[NRB][4], w[NRB][4];
      if constexpr (S::N1 > 0) {
        f4 vt[NRB];
        const FragRow<H> head = frag_head<H>(v.wr);
        Split<H> b;
        b.set(f1, one);
        frag_mul<H>(v.wr, head, b, vt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float h = h1[rb][r];
            e1[rb][r] = fmaf(-h, h, 1.f);
            ve[rb][r] = vt[rb][r] * e1[rb][r];
            w[rb][r] = ve[rb][r] * h;
          }
      }
#pragma unroll
      for (int i = 0; i < XD; ++i) {
        if (!S::has1(i)) continue;
        if (!S::has2(i)) {
          // u_i = sum_u vt[u] e1[u] zt_i[u]
          float q = 0.f;
#pragma unroll
          for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) q = fmaf(ve[rb][r], v.zt[i * H + 16 * rb + r], q);
          ur[S::col1(i)] = q * sc.ir;
          continue;
        }
        f4 Zi[NRB];
        {
          const FragRow<H> head = frag_head<H>(v.wt);
          Split<H> b;
          tangent_split<H>(v, e1, i * H, one, b);
          frag_mul<H>(v.wt, head, b, Zi);
        }
        const float iz = sc.iw * sc.ie[i];
        float q1 = 0.f, q2 = 0.f, q3 = 0.f;
#pragma unroll
        for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float zi = Zi[ob][r];
            q1 = fmaf(wd1[ob][r], zi, q1);
            q2 = fmaf(wd2[ob][r] * zi, zi, q2);
          }
        // + sum_u vt[u] h1 e1 (-2 zt_i^2) (the a1_ii column)
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) q3 = fmaf(w[rb][r], v.z2[i * H + 16 * rb + r], q3);
        ur[S::col1(i)] = q1 * iz;
        ur[S::col2(i)] = fmaf(q2 * iz, -2.f * iz, q3 * sc.ir);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    float uj[J];
#pragma unroll
    for (int c = 0; c < J; ++c) uj[c] = sum_groups(ur[c]);
    uj[0] = (uj[0] + ss[SM::BL]) * d.usd + d.umu;
#pragma unroll
    for (int c = 1; c < J; ++c) uj[c] *= d.usd;
    float wj[J], uw[J];
    if constexpr (NH == 2) {
#pragma unroll
      for (int c = 0; c < J; ++c) wj[c] = row[c];
      slot = __float_as_int(row[J + XD]);
    } else {
      window_jets<S>(xv, box, d.flag, wj);
    }
    jet_mul<S>(uj, wj, uw);
    if (valid) {
#pragma unroll
      for (int c = 0; c < J; ++c)
        if ((c & 3) == g) pairbuf[(size_t)slot * J + c] = uw[c];
    }
    if constexpr (NH == 2) {
      if (refill) {
        Team<true>::sync();   // this sub-tile's rows have been read
        put_row(xq, slotn);
      }
    }
  }
}

// Persistent forward launch: workgroup b runs the chunks of forward bin b
// in order.
// WAVE: wave w of workgroup b runs forward bin 4b + w (one-hidden-layer
// networks; a wave past the last bin has nothing to do).
template <int XD, int H, int NH, int D1M, int D2M, bool WAVE = false>
__global__ void __launch_bounds__(256, NH == 2 ? 3 : 2)
fwd_kernel(const float* __restrict__ theta, const float* __restrict__ dom, const float* __restrict__ x,
           fbpx_worklist wl, float* __restrict__ pairbuf) {
  const int bin = WAVE ? (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6) : (int)blockIdx.x;
  if (WAVE && bin >= wl.n_fbins) return;
  const int c0 = wl.fbin_chunk_start[bin], c1 = wl.fbin_chunk_start[bin + 1];
  for (int chunk = c0; chunk < c1; ++chunk) {
    if (chunk > c0) Team<WAVE>::sync();   // the team is done with the previous chunk's LDS
    fwd_chunk<XD, H, NH, D1M, D2M, WAVE>(theta, dom, x, wl, pairbuf, chunk);
  }
}

// ------------------------------------------------------------------ backward
//
// Reverse pass per pair, given gU = dL/d(segment sum of u*w jets):
//   gu = (d uw / d u)^T gU (jet_mul_T; u*w is linear in u, so u itself is not
//   needed), gur = sd_u * gu, ga_c[u] = WL[u] gur_c, dWL[u] += sum_c gur_c a2_c[u].
//   tanh-jet transpose of layer 2 (d3 = -2 (d1^2 + h d2)):
//     G_0  = d1 ga_0 + sum_i d2 z_i ga_i + sum_i (d2 z_ii + d3 z_i^2) ga_ii
//     G_i  = d1 ga_i + 2 d2 z_i ga_ii,   G_ii = d1 ga_ii
//   dW2 += sum_c G_c a1_c^T (MFMA, contraction over pairs),
//   db2 += G_0, GA_c = W2^T G_c (MFMA; registers chain),
//   layer 1 (z1_i = zt_i, z1_ii = 0):
//     gz1_0 = d1 GA_0 + sum_i d2 zt_i GA_i + sum_i d3 zt_i^2 GA_ii
//     gz1_i = d1 GA_i + 2 d2 zt_i GA_ii
//     dW1[u, k] += gz1_0 xh_k + gz1_k / sd_k,  db1 += gz1_0.
// The two-layer kernel does not form G_i and G_ii column by column: every
// linear use of the layer-1 tangents collapses into s = sum_i (gur_i a1_i +
// gur_ii a1_ii) (pair_s), so with S = W2 s and vt = W2^T (WL f1)
//   G_0 gains f2 S, the G_i a1_i^T and G_ii a1_ii^T columns of dW2 become
//   (WL f1) s^T plus 2 gur_ii WL f2 Z_i a1_i^T per second-derivative axis,
//   and GA_i = gur_i vt (+ W2^T of that axis's column), GA_ii = gur_ii vt.
// The two-layer kernel carries G~ = G / WL (row-wise; no division is
// performed: G~ is formed without the WL factor) and restores WL where G is
// consumed: W2^T G = (diag(WL) W2)^T G~ through a row-scaled LDS copy of W2,
// dW2 = diag(WL) sum_c G~_c a1_c^T and db2 = WL sum G~_0 at the end.
// Small per-unit gradients are summed over the 16 pairs of a sub-tile with
// DPP row reductions and accumulated in registers; at the end of the chunk
// everything is reduced in a fixed order (deterministic, no atomics).

// Upstream gradient of one pair w.r.t. its network output jets:
// gur = sd_u * (d uw / d u)^T gU, gU = gseg[seg] (zero for padding lanes).
template <class S>
__device__ inline void pair_upstream(const float* gU, const float* xv, const WindowBox<S::XD>& box, float flag, float usd,
                                     float* gur) {
  constexpr int J = S::J;
  float wj[J];
  window_jets<S>(xv, box, flag, wj);
  jet_mul_T<S>(gU, wj, gur);
#pragma unroll
  for (int c = 0; c < J; ++c) gur[c] *= usd;
}

// Chunk epilogue of one hidden layer: the gradient row from the waves' unit
// totals (ssmall[wave][kind][u]; kinds WL, B1, W1[:, i]) and output-bias sums
// (sbl[wave]), written out, or with ADAM applied to the subdomain's row.
// first (ADAM): the thread's first parameter and its moments, read at the
// chunk's start.
template <int XD, int H, bool WAVE = false, bool ADAM = false>
__device__ inline void finish_row(const float* ssmall, const float* sbl, int nw, float* out, float gs,
                                  const AdamFold& af, int model, const float* bc, const float* first) {
  using L = Layout<XD, H, 1>;
  using T = Team<WAVE>;
  constexpr int NS = 2 + XD;
  constexpr int K_WL = 0, K_B1 = 1, K_W1 = 2;
  const size_t r0 = (size_t)model * L::P;
  for (int i = T::tid(); i < L::P; i += T::size()) {
    float row = 0.f;
    if (i == L::BL) {
      for (int w = 0; w < nw; ++w) row += sbl[w];
    } else {
      const int at = i < L::B1 ? (K_W1 + i % XD) * H + i / XD
                               : i < L::WL ? K_B1 * H + (i - L::B1) : K_WL * H + (i - L::WL);
      for (int w = 0; w < nw; ++w) row += ssmall[w * NS * H + at];
    }
    // gs: d L / d loss for a gseg at unit upstream gradient (the row is linear
    // in gseg; 1 leaves it unchanged)
    row *= gs;
    if constexpr (!ADAM) {
      out[i] = row;
    } else {
      // the row is its subdomain's whole gradient: Adam on it in place, as
      // fbpx_adam_rows_partial updates a row from its one chunk row
      float gi = 0.f;
      gi += row;
      const bool ahead = i == T::tid();
      float p = ahead ? first[0] : af.theta[r0 + i];
      float m = ahead ? first[1] : af.mu[r0 + i];
      float v = ahead ? first[2] : af.nu[r0 + i];
      adam_elem(p, m, v, gi, bc[0], bc[1], af.k);
      af.theta[r0 + i] = p;
      af.mu[r0 + i] = m;
      af.nu[r0 + i] = v;
    }
  }
}

// [xd, h, 1]: no hidden-to-hidden layer; waves work independently.
// Bound by latency: a chunk of a training step has one to three sub-tiles, so
// the load chains and the chunk's ends weigh as much as the arithmetic.  The
// unit gradients therefore stay in registers until the chunk's end (an LDS
// read-modify-write per sub-tile and kind before), the output-bias sum is a
// wave reduction (one thread's 16 reads per wave before), and the loads run
// ahead (below): a 28-chunk step of 5,000 points 41.0 -> 37.5 us, 30 chunks of
// 1,000 points 25.7 -> 24.4, 7,022 wave chunks of 20 pairs 51.5 -> 50.8.
// WAVE: the chunk is one wave's (its own LDS copies, its slices of the
// per-wave sums).
// ADAM: bc holds the bias corrections, formed by the team's first lane in
// its first chunk (first) while the chunk's domain loads are in flight.
template <int XD, int H, int D1M, int D2M, bool WAVE = false, bool ADAM = false>
__device__ inline void bwd_one(const float* theta, const float* dom, const float* x, const fbpx_worklist& wl,
                               const float* gseg, float* partial, int chunk, float gs, const AdamFold& af,
                               float* bc, bool first = false) {
  using S = Schema<XD, D1M, D2M>;
  using L = Layout<XD, H, 1>;
  using SM = Small<XD, H, 1>;
  using T = Team<WAVE>;
  constexpr int J = S::J, NRB = H / 16, NS = 2 + XD, NT = WAVE ? 4 : 1;
  constexpr int K_WL = 0, K_B1 = 1, K_W1 = 2;
  // (with 64 units and six or seven jets in a workgroup the values ahead spill
  // inside the loop: point and jets are then read where they are used, pair
  // indices one sub-tile ahead.  [3,64,1], 3.4 million pairs: seven jets 854 ->
  // 681 us, six 652 -> 534; 690 and 577 before either)
  constexpr bool AHEAD = H < 64 || J < 6 || WAVE;
  __shared__ float ss_[NT][SM::N];
  __shared__ float ssmall_[4 * NS * H];   // per wave (four teams of one wave with WAVE)
  __shared__ float sbl_[4];
  __shared__ float szt_[NT][2 * XD * H];
  float* const ss = ss_[T::index()];
  float* const szt = szt_[T::index()];
  float* const ssmall = ssmall_ + T::index() * NS * H;
  float* const sbl = sbl_ + T::index();

  const int model = wl.chunk_model[chunk];
  const uint32_t beg = wl.chunk_start[chunk], end = wl.chunk_start[chunk + 1];
  int32_t cnt = 0;
  if constexpr (ADAM) cnt = af.count[0];   // issued with the chunk's first loads
  const float* th = theta + (size_t)model * L::P;
  const int lane = threadIdx.x & 63, wave = T::wave(), nw = T::nw();
  const int pl = lane & 15, g = lane >> 4;
  // each sub-tile's pair indices are loaded two sub-tiles ahead and its point
  // and upstream jets one ahead, so that a sub-tile waits on neither of the
  // two dependent loads; the first ones are issued around the parameter
  // staging (a chunk is often only one or two sub-tiles).  The selected index
  // is an int again: as unsigned it took five more registers with one wave per
  // chunk, [1, 32, 1] (96 -> 101: four waves per SIMD instead of five, inverse step
  // 51.3 -> 52.1 us)
  int pn, sn;
  const uint32_t k0 = beg + wave * 16 + pl, k1 = k0 + nw * 16;
  const int p0 = wl.pair_point[(int)(k0 < end ? k0 : beg)], s0 = wl.pair_seg[(int)(k0 < end ? k0 : beg)];
  if constexpr (AHEAD) {
    pn = wl.pair_point[(int)(k1 < end ? k1 : beg)];
    sn = wl.pair_seg[(int)(k1 < end ? k1 : beg)];
  } else {
    pn = p0;
    sn = s0;
  }
  SmallStage<XD, H, 1, WAVE> st;
  st.load(th);
  float xn[XD], gUn[J];
  if constexpr (AHEAD) {
#pragma unroll
    for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)p0 * XD + i];
#pragma unroll
    for (int c = 0; c < J; ++c) gUn[c] = k0 < end ? gseg[(size_t)s0 * J + c] : 0.f;
  }
  st.store(ss);
  // the row's first T::size() parameters for the update at the chunk's end
  // (one round trip less in a step of 200 points: 21.75 -> 21.5 us)
  float adam0[3] = {0.f, 0.f, 0.f};
  if constexpr (ADAM) {
    const size_t i0 = (size_t)model * L::P + (T::tid() < L::P ? T::tid() : 0);
    adam0[0] = af.theta[i0];
    adam0[1] = af.mu[i0];
    adam0[2] = af.nu[i0];
  }
  Dom d;
  load_dom(dom, model, d);
  if constexpr (ADAM) {
    if (first && T::tid() == 0) adam_bias_n(cnt, af.k, bc);
  }
  const ChunkBox<XD> box(d);
  const float* const mu = box.mu;
  const float* const isd = box.isd;
  T::sync();
  stage_zt<XD, H, SM, WAVE>(ss, isd, szt);
  T::sync();

  const LaneLds v = lane_lds<XD, H, SM>(ss, szt, ss, ss, pl, g);
  float* mysmall = ssmall + wave * NS * H;
  float dbl = 0.f, small[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) small[j] = 0.f;
  for (uint32_t base = beg + wave * 16; base < end; base += nw * 16) {
    // one wave per chunk: the weights and window tangents are read from LDS
    // per sub-tile rather than held in registers across the loop (95 VGPRs
    // instead of 120 at [1, 32, 1]: five waves per SIMD instead of four)
    if constexpr (WAVE) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // lanes past the end run the pair at beg with a zero upstream gradient
    if constexpr (!AHEAD) {
      const uint32_t k = base + pl, k1 = k + nw * 16;
#pragma unroll
      for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)pn * XD + i];
#pragma unroll
      for (int c = 0; c < J; ++c) gUn[c] = k < end ? gseg[(size_t)sn * J + c] : 0.f;
      pn = wl.pair_point[(int)(k1 < end ? k1 : beg)];
      sn = wl.pair_seg[(int)(k1 < end ? k1 : beg)];
    }
    float xv[XD], xh[XD];
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      xv[i] = xn[i];
      xh[i] = (xv[i] - mu[i]) * isd[i];
    }
    float gur[J], gU[J];
#pragma unroll
    for (int c = 0; c < J; ++c) gU[c] = gUn[c];
    if (AHEAD && base + nw * 16 < end) {
      const uint32_t kn = base + nw * 16 + pl, k2 = kn + nw * 16;
#pragma unroll
      for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)pn * XD + i];
#pragma unroll
      for (int c = 0; c < J; ++c) gUn[c] = kn < end ? gseg[(size_t)sn * J + c] : 0.f;
      pn = wl.pair_point[(int)(k2 < end ? k2 : beg)];
      sn = wl.pair_seg[(int)(k2 < end ? k2 : beg)];
    }
    pair_upstream<S>(gU, xv, box, d.flag, d.usd, gur);
    if (g == 0) dbl += gur[0];
    float h1[NRB][4];
    layer1_stream<XD, H, SM>(v, xh, h1);
    float vWL[NRB][4], gz10[NRB][4], vv[NRB][4];
    // ga_c = WL gur_c acts on layer 1 directly
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float wlu = v.vec[SM::WL + 16 * rb + r];
        const float h = h1[rb][r];
        const float d1 = tanh_d1(h), d2 = tanh_d2(h), d3 = tanh_d3(h);
        float dwl = gur[0] * h;
        float gz0 = d1 * wlu * gur[0];
#pragma unroll
        for (int i = 0; i < XD; ++i) {
          if (!S::has1(i)) continue;
          const float z = v.zt[i * H + 16 * rb + r];
          dwl = fmaf(gur[S::col1(i)], d1 * z, dwl);
          gz0 = fmaf(d2 * z, wlu * gur[S::col1(i)], gz0);
          if (S::has2(i)) {
            dwl = fmaf(gur[S::col2(i)], d2 * z * z, dwl);
            gz0 = fmaf(d3 * z * z, wlu * gur[S::col2(i)], gz0);
          }
        }
        vWL[rb][r] = dwl;
        gz10[rb][r] = gz0;
      }
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      // dW1[:, i] += gz1_0 xh_i + gz1_i / sd_i
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float t = gz10[rb][r] * xh[i];
          if (S::has1(i)) {
            const float h = h1[rb][r];
            const float z = v.zt[i * H + 16 * rb + r];
            const float wlu = v.vec[SM::WL + 16 * rb + r];
            float gzi = tanh_d1(h) * wlu * gur[S::col1(i)];
            if (S::has2(i)) gzi = fmaf(2.f * tanh_d2(h) * z, wlu * gur[S::col2(i)], gzi);
            t = fmaf(gzi, isd[i], t);
          }
          vv[rb][r] = t;
        }
      small[K_W1 + i] += reduce_units<NRB>(vv, pl);
    }
    small[K_WL] += reduce_units<NRB>(vWL, pl);
    small[K_B1] += reduce_units<NRB>(gz10, pl);
  }
  store_units<NRB, NS>(mysmall, small, H, pl, g);
  dbl = sum_row(dbl);
  if (lane == 0) sbl[wave] = dbl;
  T::sync();
  finish_row<XD, H, WAVE, ADAM>(ssmall, sbl, nw, partial + (size_t)chunk * L::P, gs, af, model, bc, adam0);
}

// dW2 accumulation.  For each gradient column c the waves write the split
// G_c and a1_c of their 16 pairs to LDS as [pair][16 units] tiles of f16 (512
// bytes per wave, 16-unit block and piece) and read them back transposed, four
// pairs of one unit per lane (ds_read_b64_tr_b16), as A (rows o) and B
// (columns u) operands of a contraction over pairs.  The four 8-byte unit
// groups of pair p are stored in the order g ^ (p >> 2): in plain order the 16
// pairs of a store phase share banks (16.3 cycles per ds_write_b64 and CU
// against 6.9), and a transposed read takes each 128-byte row of four pairs
// whole in either order (2.2 cycles).
// H = 64: the four waves run their tiles in lockstep and share one set of
// accumulators; wave w holds the quadrant of row blocks 2 (w >> 1) + {0, 1}
// and column blocks 2 (w & 1) + {0, 1} and contracts it over the pairs of all
// four waves (the whole 64 x 64 set would not fit a wave's registers), with
// workgroup barriers around each column.
// H <= 32 (PRIV): every wave holds all NRB^2 blocks (16 registers at H = 32)
// over its own pairs, reading back only what it wrote itself, so the tile
// loop needs no workgroup barrier: LDS operations of one wavefront are
// performed in order, and a wavefront-scope fence keeps the compiler from
// moving the reads above the writes (or the next writes above the reads).
template <int H>
struct DW2Own {
  static constexpr int NRB = H / 16;
  static constexpr bool PRIV = H <= 32;
  static constexpr int NOB = PRIV ? NRB * NRB : 4;  // blocks held by a wave
  static constexpr int TILE = 128;                  // floats of a wave's tile (16 pairs x 16 units, one piece)
  static constexpr int BS = 4 * TILE;               // of a 16-unit block (four waves)
  static constexpr int PS = NRB * BS;               // of a piece
  static constexpr int TSZ = 2 * PS;                // of a buffer
  // float offset in a tile of pair p, units 4 g .. 4 g + 3
  __device__ static int at(int p, int g) { return 8 * p + 2 * (g ^ (p >> 2)); }
  // the address lane 16 q + s supplies to a transposed read, which gives it
  // unit s of pairs 4 q .. 4 q + 3
  __device__ static int at_tr(int lane) { return at(lane >> 2, lane & 3); }
  __device__ static int row_block(int wave, int j) { return PRIV ? j / NRB : 2 * (wave >> 1) + (j >> 1); }
  __device__ static int col_block(int wave, int j) { return PRIV ? j % NRB : 2 * (wave & 1) + (j & 1); }
};

// Orders a wave's LDS tiles around the dW2 reads: a workgroup barrier
// when the waves share the accumulators, else a wavefront-scope fence.
template <bool PRIV>
__device__ inline void tile_sync() {
  if constexpr (PRIV)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  else
    __syncthreads();
}

__device__ inline h4v read_tr(const float* p) {
  typedef __fp16 hh4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) hh4* lds_h4;
  return __builtin_bit_cast(h4v, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4)p));
}
__device__ inline h8v join(h4v a, h4v b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// dW2 += G_c a1_c^T over this wave's own 16 pairs (PRIV), all NRB^2 blocks;
// gt, at: this wave's tiles at its lane offset.  hi and lo of G side by side
// in a K of 32 against lo of a1 twice (which adds the lo lo product) and hi
// of a1 twice.
template <int H>
__device__ inline void dw2_private(const float* gt, const float* at, f4* dW2) {
  using O = DW2Own<H>;
  constexpr int NRB = H / 16;
  h4v ah[NRB], al[NRB], bh[NRB], bl[NRB];
#pragma unroll
  for (int b = 0; b < NRB; ++b) {
    ah[b] = read_tr(gt + b * O::BS);
    al[b] = read_tr(gt + O::PS + b * O::BS);
    bh[b] = read_tr(at + b * O::BS);
    bl[b] = read_tr(at + O::PS + b * O::BS);
  }
#pragma unroll
  for (int j = 0; j < O::NOB; ++j) {
    const h8v a = join(ah[j / NRB], al[j / NRB]);
    dW2[j] = mfma_k32(a, join(bl[j % NRB], bl[j % NRB]), dW2[j]);
    dW2[j] = mfma_k32(a, join(bh[j % NRB], bh[j % NRB]), dW2[j]);
  }
}

// dW2[j] += G_c a1_c^T over the tile's 64 pairs (two K-steps of two waves'
// pairs), this wave's quadrant; gt, at: the quadrant's first row / column
// block at the lane offset.
template <int H>
__device__ inline void dw2_shared(const float* gt, const float* at, f4* dW2) {
  using O = DW2Own<H>;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    h8v a[2][2], b[2][2];   // [block][piece]
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int o = c * O::PS + j * O::BS + 2 * ks * O::TILE;
        a[j][c] = join(read_tr(gt + o), read_tr(gt + o + O::TILE));
        b[j][c] = join(read_tr(at + o), read_tr(at + o + O::TILE));
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dW2[j] = mfma_k32(a[j >> 1][1], b[j & 1][0], dW2[j]);
      dW2[j] = mfma_k32(a[j >> 1][0], b[j & 1][1], dW2[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) dW2[j] = mfma_k32(a[j >> 1][0], b[j & 1][0], dW2[j]);
  }
}

// Write this wave's split values (units x 16 pairs) to its tiles of a buffer;
// tl = buffer + wave TILE + at(pl, g).
template <int H>
__device__ inline void store_tile(float* tl, const Split<H>& v) {
  using O = DW2Own<H>;
#pragma unroll
  for (int b = 0; b < H / 16; ++b) {
    *reinterpret_cast<u2v*>(tl + b * O::BS) = u2v{v.hi[2 * b], v.hi[2 * b + 1]};
    *reinterpret_cast<u2v*>(tl + O::PS + b * O::BS) = u2v{v.lo[2 * b], v.lo[2 * b + 1]};
  }
}

// This thread's largest |gseg| per jet column over its share of the chunk's
// pairs (stage_two reduces them over the workgroup), in two halves so that the
// other loads of the chunk's start go between them: indices() issues the loads
// of the first FIRST segment indices, values() the rows'.
template <int J>
struct GradientMax {
  static constexpr int FIRST = 4;
  int seg[FIRST];
  float m[J];
  __device__ void indices(const fbpx_worklist& wl, uint32_t beg, uint32_t end) {
#pragma unroll
    for (int j = 0; j < FIRST; ++j) {
      const uint32_t k = beg + threadIdx.x + 256 * j;
      seg[j] = wl.pair_seg[k < end ? k : beg];   // a repeated pair does not change the maximum
    }
  }
  __device__ void values(const fbpx_worklist& wl, const float* gseg, uint32_t beg, uint32_t end) {
#pragma unroll
    for (int c = 0; c < J; ++c) m[c] = 0.f;
#pragma unroll
    for (int j = 0; j < FIRST; ++j)
#pragma unroll
      for (int c = 0; c < J; ++c) m[c] = fmaxf(m[c], fabsf(gseg[(size_t)seg[j] * J + c]));
#pragma unroll 4
    for (uint32_t k = beg + threadIdx.x + 256 * FIRST; k < end; k += 256) {
      const int sk = wl.pair_seg[k];
#pragma unroll
      for (int c = 0; c < J; ++c) m[c] = fmaxf(m[c], fabsf(gseg[(size_t)sk * J + c]));
    }
  }
};

// [xd, h, h, 1]: hidden-to-hidden layer on MFMA, streamed one axis at a time.
// Scales (all powers of two, Scales): everything linear in the upstream
// gradient is carried times 2^k and the tile's sign; on top of it (marked ' below)
//   Z_i' = Z_i 2^(w + e[i]),  S' = S 2^w, and with them G_0', dWL', Q' times 2^w;
//   vt' = vt 2^r and gz1_0' times 2^r (over -2 e1 until column 0);  stored G_i times 2^-e[i], so that
//   G_i (e1 zt_i 2^e[i])^T adds to dW2 like the other columns, and so
//   GA_i' and gz1_i' carry 2^(r - e[i]).
template <int XD, int H, int D1M, int D2M>
__device__ inline void bwd_two(const float* theta, const float* dom, const float* x, const fbpx_worklist& wl,
                               const float* gseg, float* partial, int chunk, float gs) {
  using S = Schema<XD, D1M, D2M>;
  using L = Layout<XD, H, 2>;
  using SM = Small<XD, H, 2>;
  using O = DW2Own<H>;
  using R = PairRows;
  constexpr int J = S::J, NRB = H / 16, NS = 3 + XD;
  constexpr int K_WL = 0, K_B1 = 1, K_W1 = 2, K_B2 = 2 + XD;
  // H <= 32 and XD <= 2 (wave-private dW2, registers to spare): the small
  // per-unit gradients but dWL (dW1, db1, db2) are summed per lane over the
  // chunk's tiles and reduced over the pair lanes once per chunk instead of
  // once per tile (with three axes the unrolled axis loop would spill; with
  // dWL as well, 13 more spilled registers and 154 us against 148.5)
  constexpr bool ACC = DW2Own<H>::PRIV && XD <= 2;
  constexpr int AXIS_UNROLL = H == 64 || ACC ? XD : 1;
  static_assert(H >= 16 && H <= 64, "hidden width 16, 32 or 64");
  __shared__ float ss[SM::N];
  __shared__ float szt[3 * XD * H];
  __shared__ __attribute__((aligned(16))) float swt[2 * W2Frags<H>::SET];
  float* const swr = swt + W2Frags<H>::SET;
  __shared__ __attribute__((aligned(16))) float strans[2 * O::TSZ];
  // per wave: its pair rows, and at the chunk's end its unit totals
  constexpr int SW = R::WAVE > NS * H ? R::WAVE : NS * H;
  __shared__ __attribute__((aligned(16))) float srow[4 * SW];
  __shared__ float sbl[4];
  float* sta = strans;            // a1 columns
  float* stg = strans + O::TSZ;   // G columns

  const int model = wl.chunk_model[chunk];
  const uint32_t beg = wl.chunk_start[chunk], end = wl.chunk_start[chunk + 1];
  const float* th = theta + (size_t)model * L::P;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int pl = lane & 15, g = lane >> 4;
  // the index loads of the gradient maxima and of the first tile, ahead of
  // everything that waits
  GradientMax<J> gmax;
  gmax.indices(wl, beg, end);
  const uint32_t k0 = beg + wave * 16 + g * 64 + pl;   // the pair of this lane's first row
  const int p0 = wl.pair_point[k0 < end ? k0 : beg], seg0 = wl.pair_seg[k0 < end ? k0 : beg];
  Dom d;
  load_dom(dom, model, d);
  const ChunkBox<XD> box(d);
  const float* const mu = box.mu;
  const float* const isd = box.isd;
  const float one = opaque_one();
  Scales<XD> sc;
  float x0[XD], gU0[J];   // the first row's point and upstream jets
  stage_two<S, H, SM, true, true>(
      th, d, isd,
      [&]() -> const float* {
#pragma unroll
        for (int i = 0; i < XD; ++i) x0[i] = x[(size_t)p0 * XD + i];
#pragma unroll
        for (int c = 0; c < J; ++c) gU0[c] = k0 < end ? gseg[(size_t)seg0 * J + c] : 0.f;
        gmax.values(wl, gseg, beg, end);
        return gmax.m;
      },
      one, ss, szt, swt, swr, srow, sc);
  d.usd = uniform(d.usd * sc.k);
  // The f16 matrix instructions align their products by cutting them off
  // towards minus infinity: a product of split operands comes out about 5e-9 of
  // its typical size too small, always on the same side (the float32
  // instruction: none).  Added over a subdomain's pairs, whose upstream
  // gradients differ in sign, that offset grows with their number N and the
  // gradient with its root: 2.4e-7 of it at N = 3,600.  Everything linear in the
  // upstream gradient is therefore carried with the other sign in every second
  // tile (and every second chunk starts with it), and the signs are taken off
  // where the tiles are added up.  Of the tile's cost only the dW2 accumulators'
  // change of sign is new: wave step as before, Burgers slab step 126.6 -> 127.7 us,
  // Poisson step 247.7 -> 250.7.
  const float lane_sign = ((g + chunk) & 1) ? -1.f : 1.f;   // of this lane's rows: tiles g, g + 4, ...

  // WL of the unit a reduction leaves in this lane (for G_0')
  const float wl_red = ss[SM::WL + 16 * (pl >> 2) + 4 * g + (pl & 3)] * sc.iw;
  const LaneLds v = lane_lds<XD, H, SM>(ss, szt, swt, swr, pl, g);
  float* const staw = sta + wave * O::TILE + O::at(pl, g);   // this wave's stores
  float* const stgw = stg + wave * O::TILE + O::at(pl, g);
  // dW2 reads: this wave's own tiles (PRIV) or its quadrant's blocks
  const float* const star = sta + (O::PRIV ? wave * O::TILE : O::col_block(wave, 0) * O::BS) + O::at_tr(lane);
  const float* const stgr = stg + (O::PRIV ? wave * O::TILE : O::row_block(wave, 0) * O::BS) + O::at_tr(lane);
  float aW1[ACC ? XD : 1][NRB][4], aB1[NRB][4], aB2[NRB][4];
  if constexpr (ACC) {
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int i = 0; i < XD; ++i) aW1[i][rb][r] = 0.f;
        aB1[rb][r] = aB2[rb][r] = 0.f;
      }
  }
  f4 dW2[O::NOB];
#pragma unroll
  for (int j = 0; j < O::NOB; ++j) dW2[j] = f4{0.f, 0.f, 0.f, 0.f};
  float dbl = 0.f;
  // !ACC: this lane's unit totals over the chunk (reduce_units), by kind
  float small[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) small[j] = 0.f;

  // with shared dW2 blocks every wave runs the same number of tiles (barriers
  // below); with wave-private blocks (H <= 32) a wave runs only the tiles in
  // which its 16-pair sub-tile holds a pair of the chunk.  Lanes past the
  // chunk end carry zero upstream gradient and so contribute nothing.
  const int ntile =
      (int)(O::PRIV ? __builtin_amdgcn_readfirstlane((end - beg + (63 - 16 * wave)) >> 6) : (end - beg + 63) >> 6);
  // this lane's row (upstream gradient, normalised point) of the next four
  // tiles.  Their points and upstream jets are fetched during the tile
  // before (indices at the start of its column-0 phase, data before its last
  // dW2 column), so the two dependent global loads do not stall a tile's start
  static_assert(J + XD <= R::ROW, "a pair's row");
  float* const rows = srow + wave * SW;
  const auto put_row = [&](const float* xp, const float* gU) {
    float gur[J];
    pair_upstream<S>(gU, xp, box, d.flag, d.usd * lane_sign, gur);
    dbl += gur[0];
    float* const to = rows + lane * R::ROW;
#pragma unroll
    for (int c = 0; c < J; ++c) to[c] = gur[c];
#pragma unroll
    for (int i = 0; i < XD; ++i) to[J + i] = (xp[i] - mu[i]) * isd[i];
    Team<true>::sync();
  };
  put_row(x0, gU0);
  for (int t = 0; t < ntile; ++t) {
    const float sign = ((t + chunk) & 1) ? -1.f : 1.f;
#pragma unroll
    for (int j = 0; j < O::NOB; ++j) dW2[j] = -dW2[j];
    const float* const row = rows + ((t & 3) * 16 + pl) * R::ROW;
    float gur[J], xh[XD];
#pragma unroll
    for (int c = 0; c < J; ++c) gur[c] = row[c];
#pragma unroll
    for (int i = 0; i < XD; ++i) xh[i] = row[J + i];
    const bool refill = (t & 3) == 3 && t + 1 < ntile;

    float h1[NRB][4];
    layer1_stream<XD, H, SM>(v, xh, h1);
    float vWL[NRB][4], gz10[NRB][4], vv[NRB][4];

    // ---- Z_0 = W2 h1 + b2 -> h2
    float h2[NRB][4];
    {
      f4 Z0[NRB];
      layer2_value<H, SM>(v, h1, one, Z0);
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) h2[ob][r] = tanh_f(Z0[ob][r], sc.iw);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- S = W2 s,  G_S = f1,  vt = W2~^T G_S (d L / d s),  dW2 += G_S s^T
    //      (column S first, so that s is dead before the axes).  With
    //      Q = sum_i gur_ii Z_i^2 (accumulated per axis):
    //        G_0 = f1 gur_0 + f2 S + f3 Q,  dWL = gur_0 h2 + f1 S + f2 Q
    //      (f1 = 1 - h2^2, f2 = -2 h2 f1, f3 = f1 (4 - 6 f1)).  The layer-1
    //      gradient starts as gz1_0 = vt rv (see pair_s); the axes add
    //      e2 zt_i GA_i and column 0 adds e1 GA_0.
    float G0[NRB][4];
    f4 vt[NRB];
    float Sx[NRB][4], Q[NRB][4];
    const float gur0 = gur[0] * sc.w;
    if constexpr (S::N1 == 0) {
      // value only: no tangents, s = 0
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float h = h2[ob][r];
          G0[ob][r] = fmaf(-h, h, 1.f) * gur0;
          vWL[ob][r] = gur0 * h;
          gz10[ob][r] = 0.f;
        }
    } else {
      float rv[NRB][4];
      Split<H> ssp, fsp;
      {
        const FragRow<H> head = frag_head<H>(v.wt);
        {
          float sv[NRB][4];
          pair_s<S, H>(v, h1, gur, sv, rv);
          ssp.set(sv, one);
        }
        f4 Sv[NRB];
        frag_mul<H>(v.wt, head, ssp, Sv);
#pragma unroll
        for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            Sx[ob][r] = Sv[ob][r];
            Q[ob][r] = 0.f;
          }
      }
      const FragRow<H> head = frag_head<H>(v.wr);
      {
        float f1[NRB][4];
#pragma unroll
        for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
          for (int r = 0; r < 4; ++r) f1[ob][r] = fmaf(-h2[ob][r], h2[ob][r], 1.f);
        fsp.set(f1, one);
      }
      tile_sync<O::PRIV>();   // the previous tile's column has been consumed
      store_tile<H>(staw, ssp);
      store_tile<H>(stgw, fsp);
      frag_mul<H>(v.wr, head, fsp, vt);
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) gz10[rb][r] = vt[rb][r] * rv[rb][r];
      tile_sync<O::PRIV>();
      if constexpr (O::PRIV)
        dw2_private<H>(stgr, star, dW2);
      else
        dw2_shared<H>(stgr, star, dW2);
    }
    // from here on layer 1 enters through h1 and e1 = 1 - h1^2, and the axes
    // take layer 2 through p2 = -4 h2 (1 - h2^2) = 2 f2
    float e1[NRB][4], p2[NRB][4];
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        e1[rb][r] = fmaf(-h1[rb][r], h1[rb][r], 1.f);
        p2[rb][r] = (-4.f * h2[rb][r]) * fmaf(-h2[rb][r], h2[rb][r], 1.f);
      }
    __builtin_amdgcn_sched_barrier(0);

    // ---- per axis.  d L / d a1_i = gur_i vt (+ W2~^T G_i when the axis has a
    //      second derivative), d L / d a1_ii = gur_ii vt;  G_i = 2 gur_ii f2 Z_i
    //        gz1_i = e1 (gur_i vt + GA_i) + 2 gur_ii e2 zt_i vt,
    //        gz1_0 += e2 zt_i GA_i.
    //      Unrolled at h = 64; a real loop below that (one register allocation
    //      serves every axis), which the compiler allocates with fewer spills.
#pragma unroll AXIS_UNROLL
    for (int i = 0; i < XD; ++i) {
      if (!S::has1(i)) continue;
      const bool two = S::has2(i);
      const float gur_a = pick<J>(gur, S::col1(i));
      const float gur_b = two ? pick<J>(gur, S::col2(i)) : 0.f;
      const float e_i = pick<XD>(sc.e, i), ie_i = pick<XD>(sc.ie, i);
      // gz1_i' = gz1_i 2^(r - e[i]) (r alone without a second derivative)
      const float post = pick<XD>(isd, i) * (sc.ir * sign) * (two ? e_i : 1.f);
      const int zrow = i * H;
      float gzi[NRB][4];
      if (two) {
        Split<H> gsp, asp;
        FragRow<H> head = frag_head<H>(v.wt);
        tangent_split<H>(v, e1, zrow, one, asp);
        {
          f4 Zi[NRB];
          frag_mul<H>(v.wt, head, asp, Zi);
          head = frag_head<H>(v.wr);
          const float gq = (gur_b * ie_i) * (sc.iw * ie_i);   // Q' += gur_b Z_i^2 2^w
          float Gi[NRB][4];
#pragma unroll
          for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float z = Zi[ob][r], t = gq * z;
              Q[ob][r] = fmaf(t, z, Q[ob][r]);
              Gi[ob][r] = p2[ob][r] * t;                      // 2 gur_b f2 Z_i 2^-e[i]
            }
          gsp.set(Gi, one);
        }
        __builtin_amdgcn_sched_barrier(0);
        // column i: publish G_i and a1_i, then W2~^T G_i while the other waves
        // catch up
        tile_sync<O::PRIV>();
        store_tile<H>(staw, asp);
        store_tile<H>(stgw, gsp);
        {
          f4 GA[NRB];
          frag_mul<H>(v.wr, head, gsp, GA);
          const float gb4 = -4.f * gur_b * ie_i * ie_i, ga = gur_a * ie_i;
#pragma unroll
          for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float y = h1[rb][r] * v.zs[zrow + 16 * rb + r];   // -e2 zt_i 2^e[i] / (2 e1)
              gzi[rb][r] = e1[rb][r] * fmaf(vt[rb][r], fmaf(gb4, y, ga), GA[rb][r]);
              gz10[rb][r] = fmaf(y, GA[rb][r], gz10[rb][r]);
            }
        }
        tile_sync<O::PRIV>();
        if constexpr (O::PRIV)
          dw2_private<H>(stgr, star, dW2);
        else
          dw2_shared<H>(stgr, star, dW2);
      } else {
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) gzi[rb][r] = e1[rb][r] * (gur_a * vt[rb][r]);
      }
      // dW1[:, i] through z1_i = zt_i (the 1 / sd_i factor after the sum)
      if constexpr (ACC) {
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) aW1[i][rb][r] = fmaf(gzi[rb][r], post, aW1[i][rb][r]);
      } else {
        {
          const float r = reduce_units<NRB>(gzi, pl) * post;
#pragma unroll
          for (int j = 0; j < XD; ++j) small[K_W1 + j] += j == i ? r : 0.f;
        }
      }
    }
    if constexpr (S::N1 > 0) {
      opaque<NRB>(h2);
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // G_0 = f1 (gur_0 - 2 h2 S + (4 - 6 f1) Q), dWL = gur_0 h2 + f1 (S - 2 h2 Q)
          const float h = h2[ob][r];
          const float f1 = fmaf(-h, h, 1.f), m = -2.f * h;
          G0[ob][r] = f1 * fmaf(m, Sx[ob][r], fmaf(fmaf(-6.f, f1, 4.f), Q[ob][r], gur0));
          vWL[ob][r] = fmaf(f1, fmaf(m, Q[ob][r], Sx[ob][r]), gur0 * h);
        }
    }
    // ---- column 0: db2 += G_0, dW2 += G_0 h^T, W2~^T G_0 -> layer 1
    // (h = 64 reads in every tile what the fourth uses: a branch here splits the
    // tile's schedule, 78 -> 259 registers spilled, 3,360 -> 10,070 us; below it
    // the branch is the cheaper form)
    const uint32_t kn = beg + ((uint32_t)(t | 3) + 1 + g) * 64 + wave * 16 + pl;   // the next row's pair
    const bool valid_n = kn < end;
    const bool fetch = !O::PRIV || refill;
    int pn, segn;
    if (fetch) {
      pn = wl.pair_point[valid_n ? kn : beg];
      segn = wl.pair_seg[valid_n ? kn : beg];
    }
    if constexpr (ACC) {
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) aB2[ob][r] = fmaf(G0[ob][r], sign, aB2[ob][r]);
    } else {
      small[K_B2] = fmaf(reduce_units<NRB>(G0, pl), wl_red * sign, small[K_B2]);
    }
    {
      Split<H> gsp, hsp;
      const FragRow<H> head = frag_head<H>(v.wr);
#pragma unroll
      for (int ob = 0; ob < NRB; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) G0[ob][r] *= sc.iw;
      gsp.set(G0, one);
      hsp.set(h1, one);
      tile_sync<O::PRIV>();
      store_tile<H>(staw, hsp);
      store_tile<H>(stgw, gsp);
      f4 GA[NRB];
      frag_mul<H>(v.wr, head, gsp, GA);
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) gz10[rb][r] = e1[rb][r] * fmaf(-2.f, gz10[rb][r], GA[rb][r]);
    }
    small[K_WL] = fmaf(reduce_units<NRB>(vWL, pl), sc.iw * sign, small[K_WL]);
    // dW1[:, i] += gz1_0 xh_i (the gz1_i parts were added per axis)
    if constexpr (ACC) {
      float xr[XD];
#pragma unroll
      for (int i = 0; i < XD; ++i) xr[i] = xh[i] * (sc.ir * sign);
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int i = 0; i < XD; ++i) aW1[i][rb][r] = fmaf(gz10[rb][r], xr[i], aW1[i][rb][r]);
          aB1[rb][r] = fmaf(gz10[rb][r], sign, aB1[rb][r]);
        }
    } else {
#pragma unroll
      for (int i = 0; i < XD; ++i) {
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) vv[rb][r] = gz10[rb][r] * xh[i];
        small[K_W1 + i] = fmaf(reduce_units<NRB>(vv, pl), sc.ir * sign, small[K_W1 + i]);
      }
      small[K_B1] = fmaf(reduce_units<NRB>(gz10, pl), sc.ir * sign, small[K_B1]);
    }
    // the next row's point and upstream jets, in flight during the last dW2 column
    __builtin_amdgcn_sched_barrier(0);
    float xn[XD], gUn[J];
    if (fetch) {
#pragma unroll
      for (int i = 0; i < XD; ++i) xn[i] = x[(size_t)pn * XD + i];
#pragma unroll
      for (int c = 0; c < J; ++c) gUn[c] = valid_n ? gseg[(size_t)segn * J + c] : 0.f;
    }
    tile_sync<O::PRIV>();
    if constexpr (O::PRIV)
      dw2_private<H>(stgr, star, dW2);
    else
      dw2_shared<H>(stgr, star, dW2);
    // (the next tile's first column has a barrier before its stores)
    if (refill) put_row(xn, gUn);
  }

  // ---- end of chunk: the gradient row from the waves' sums
  if constexpr (ACC) {
#pragma unroll
    for (int i = 0; i < XD; ++i) small[K_W1 + i] = reduce_units<NRB>(aW1[i], pl);
    small[K_B1] = reduce_units<NRB>(aB1, pl) * sc.ir;
    small[K_B2] = reduce_units<NRB>(aB2, pl) * wl_red;
  }
  store_units<NRB, NS>(rows, small, H, pl, g);   // after this wave's last row
  dbl = sum_groups(sum_row(dbl * lane_sign));
  if (lane == 0) sbl[wave] = dbl;
  __syncthreads();   // every wave is done with the tiles
  // H = 64: the waves hold disjoint dW2 blocks; H <= 32: every wave holds every
  // block over its own pairs, one copy per wave, summed in wave order below
  constexpr int NC = O::PRIV ? 4 : 1;
  static_assert(NC * H * H <= 2 * O::TSZ, "the dW2 copies reuse the tile buffers");
  {
    float* const sw = strans + (O::PRIV ? wave * H * H : 0);
    const float last_sign = ((ntile - 1 + chunk) & 1) ? -1.f : 1.f;
#pragma unroll
    for (int j = 0; j < O::NOB; ++j) {
      const int ob = O::row_block(wave, j);
      const int col = 16 * O::col_block(wave, j) + pl;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sw[(16 * ob + 4 * g + r) * H + col] = dW2[j][r] * (v.vec[SM::WL + 16 * ob + r] * last_sign);
    }
  }
  __syncthreads();
  float* const out = partial + (size_t)chunk * L::P;
  for (int i = threadIdx.x; i < H * H; i += 256) {
    float s = strans[i];
#pragma unroll
    for (int w = 1; w < NC; ++w) s += strans[w * H * H + i];
    out[L::W2 + i] = s * sc.ik * gs;   // in this order: sc.ik gs alone may overflow
  }
  for (int t = threadIdx.x; t < NS * H; t += 256) {
    const int kind = t / H, u = t % H;
    const float s = (srow[t] + srow[SW + t]) + (srow[2 * SW + t] + srow[3 * SW + t]);
    const int dst = kind == K_WL ? L::WL + u : kind == K_B1 ? L::B1 + u : kind == K_B2 ? L::B2 + u
                                                                       : L::W1 + u * XD + (kind - K_W1);
    out[dst] = s * sc.ik * gs;
  }
  if (threadIdx.x == 0) out[L::BL] = ((sbl[0] + sbl[1]) + (sbl[2] + sbl[3])) * sc.ik * gs;
}

// g_scale: NULL, or d L / d loss when gseg holds the segment gradients at
// unit upstream gradient; it multiplies each chunk's gradient row as the row
// is written (finish_row).
// ADAM (one-hidden-layer networks): every trained subdomain row is one
// chunk, and each chunk's row is applied to theta by Adam (af) in place of
// being written to partial; the team (workgroup, or wave with WAVE) that
// finishes last advances the count.
template <int XD, int H, int NH, int D1M, int D2M, bool WAVE = false, bool ADAM = false>
__global__ void __launch_bounds__(256, 2)
bwd_kernel(const float* __restrict__ theta, const float* __restrict__ dom, const float* __restrict__ x,
           fbpx_worklist wl, const uint8_t* __restrict__ chunk_train, const float* __restrict__ gseg,
           const float* __restrict__ g_scale, float* __restrict__ partial, AdamFold af) {
  static_assert(!WAVE || NH == 1, "one wave per chunk: one-hidden-layer networks");
  static_assert(!ADAM || NH == 1, "the folded optimizer step: one-hidden-layer networks");
  const float gs = g_scale ? g_scale[0] : 1.f;
  // the bias corrections, formed in LDS by each team in its first chunk from
  // the count as it reads it before the last team advances it (the read
  // completes before the team's own count below), read where a row is
  // applied (after the chunk's barriers)
  __shared__ float sbc[2];
  bool first = true;
  // persistent: workgroup b runs the chunks of backward bin b in order (WAVE:
  // wave w runs bin 4b + w)
  const int bin = WAVE ? (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6) : (int)blockIdx.x;
  if (WAVE && bin >= wl.n_bbins) return;
  const int c0 = wl.bbin_chunk_start[bin], c1 = wl.bbin_chunk_start[bin + 1];
  for (int chunk = c0; chunk < c1; ++chunk) {
    if (chunk_train != nullptr && chunk_train[chunk] == 0) continue;
    Team<WAVE>::sync();   // the team is done with the previous chunk's LDS
    if constexpr (NH == 1)
      bwd_one<XD, H, D1M, D2M, WAVE, ADAM>(theta, dom, x, wl, gseg, partial, chunk, gs, af, sbc, first);
    else
      bwd_two<XD, H, D1M, D2M>(theta, dom, x, wl, gseg, partial, chunk, gs);
    first = false;
  }
  if constexpr (ADAM) {
    if (Team<WAVE>::tid() == 0 && atomicAdd(af.count_done, 1) == wl.n_bbins - 1) {
      atomicAdd(af.count, 1);
      atomicExch(af.count_done, 0);
    }
  }
}

}  // namespace fbpx
