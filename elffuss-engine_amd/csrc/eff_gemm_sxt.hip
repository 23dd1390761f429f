// Split-x product over LDS-shared tiles, for prompts of the K and IQ types:
// the arithmetic of eff_gemm_sx.hip (x as fp16 hi and lo parts, integer weights
// exact in fp16, f32 sums, one scale per block of 256), from the same prepared
// x, for token counts where reading x bounds that kernel.
//
// What bounds k_sx at many tokens: every wave reads its x fragments from L2 by
// itself, 0.5 KB per matrix instruction with 64 rows per wave: 64 bytes per
// clock and CU with the matrix cores busy, all that a CU's vector memory path
// delivers. Here a workgroup's waves share x through LDS.
//
// Workgroup: 8 waves (2 per SIMD) over 64 tokens x 128 rows, as 4 groups of 32
// rows x 2 slices of k (slice z takes every second block of 256). A wave holds 2
// tiles of 32 tokens x 32 rows: per step of 16 k it reads 2 lo and 2 hi fragments
// of x (4 KB) for 4 v_mfma_f32_32x32x16_f16, decodes its weight fragment in
// registers, and adds lo and hi into accumulators of their own,
//   D2 += u lo, D += u hi,
// folded once per block: acc += (D + D2) d p (p: x's block scales). x flows in
// groups of 4 steps through two LDS buffers (direct-to-LDS loads a group ahead,
// one barrier per group); the raw weights of the next block are loaded into a
// region of LDS of the wave's own while the present block's are in registers.
//
// Errors against 64 bits are k_sx's or smaller, for weights of both signs and of
// one (normal, |normal|, exponential and its cube, -|normal|, normal + 1 sigma) and
// for x of both signs and of one, k = 512 to 14336. What it takes (relative L2, k =
// 2048, normal x; k_sx / here):
//  - Q4_K and Q2_K multiply u = sc (q - c) instead of sc q, c the block's zero as
//    its minima put it (near dmin sum mn / (d sum sc): about half the range for
//    weights of both signs, 0 where there are no minima), and D opens with the
//    group sums' terms, -(dmin / d) sum mn_g S_g + c sum sc_g S_g: sums near those
//    of the weights themselves. Normal weights 3.15e-7 / 1.46e-7 (Q4_K) and
//    2.00e-7 / 1.42e-7 (Q2_K), |normal| 1.24e-7 / 1.04e-7 and 0.89e-7 / 0.84e-7, the
//    cube of exponential 0.93e-7 / 0.86e-7 and 0.76e-7 / 0.76e-7. With c fixed at
//    the middle of the range and lo in D, weights of one sign came to up to 4.5e-7.
//  - A block's hi parts in two sums of 8 steps (not IQ2_XXS: 1.30e-7 both ways), the
//    blocks in four runs.
// A wave of 64 rows halves the reads of x, but with lo in accumulators of its own it
// leaves registers for one wave per SIMD (us, Q4_K, 64 rows / 32: 8192 x 2048 at 512
// tokens 53.8 / 54.6, 14336 x 4096 at 512 177 / 170): 0.4% over 199 shapes.
//
// Q6_K: u = sc (q - 32) has up to 13 bits, so its fp16 rounding v = fp16(u) is
// off by r = u - v in {-1, 0, 1}, and only where |u| > 2048. The product takes
// hi and lo times v, hi times r, and, below 8 blocks of k, lo times r (below 2^-22
// of the term). Left out there it shows (weights of both signs: 1.04 of k_sx's error
// at k = 512 and 1.03 at 1024, with it 1.00 and 0.99, 0.98 at 1792); from 8 blocks
// the shorter chains of sums make up for it (1.00 at 2048, of one sign up to 1.03;
// 0.88-0.91 at 2304, 0.71-0.73 at 8192). It costs a fourth matrix instruction (8192 x
// 2048 at 512 tokens 62.9 / 69.7 us, k_sx 130). One fold per block instead of 16, whose
// 24 vector instructions per matrix instruction bound k_sx there.
//
// What bounds it: no unit (Q4_K 8192 x 2048 at 512 tokens: matrix cores busy 37% of
// the kernel's clocks at 1.9 GHz, vector instructions 41%, LDS 27%, L2 10 TB/s). A CU
// holds one workgroup, and nothing covers its first loads (about 4 us), the barrier
// per group, the chain at a block's start and its end. us, k_sx and this kernel, both
// with the preparation of x: Q4_K 8192 x 2048 at 512 tokens 72.1 / 56.4, at 1000 150.0 /
// 107.2, Q6_K 2048 x 8192 at 300 78.0 / 50.4.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/elffuss_amd.h"
#include "eff_device.h"
#include "eff_formats.h"
#include "eff_kernels.h"
#include "eff_sx.h"

namespace eff {

static __constant__ uint64_t c_grid_sxt[256] = {
#include "iq2xxs_grid.inc"
};

namespace {

// The raw weights of 32 rows, unit by unit (a block of 256 weights, or half of
// one): NI direct-to-LDS loads of 1 KB, whose lane (row j, half h) brings 16
// bytes; 16-byte piece P of row j is then at 512 P + 16 j of the region. `fetch`
// issues the loads of unit `un` of the block at byte `bo` of the lane's row,
// `take` reads the unit's weights into registers, `step` decodes the 8 weights
// of the lane in step s of the unit (k 16 s + 8 h .. + 7) to exact fp16.
template <int TYPE> struct SxtW;

__device__ __forceinline__ uint64_t lds64(const uint8_t *p) { return *(const uint64_t *)p; }
__device__ __forceinline__ uint32_t lds32(const uint8_t *p) { return *(const uint32_t *)p; }

// 8 bytes b (v0, v1) -> (1024 + b) (sc f) + sc o as fp16: every operand and the
// result are exact, so the fused multiply-add is.
__device__ __forceinline__ half8 dec_centred(uint32_t v0, uint32_t v1, uint32_t sc, float f, float o) {
  const _Float16 s = (_Float16)((float)sc * f), c = (_Float16)((float)sc * o);
  const half2v s2 = {s, s}, c2 = {c, c};
  const half2v a = __builtin_elementwise_fma(h1024_lo(v0), s2, c2);
  const half2v b = __builtin_elementwise_fma(h1024_hi(v0), s2, c2);
  const half2v e = __builtin_elementwise_fma(h1024_lo(v1), s2, c2);
  const half2v g = __builtin_elementwise_fma(h1024_hi(v1), s2, c2);
  return half8{a.x, a.y, b.x, b.y, e.x, e.y, g.x, g.y};
}

// The block's scale d and the ratio its minima's sums are scaled by. A block
// with d = 0 keeps its minima: its u are zeroed (by the caller) and the scale is
// dmin itself.
__device__ __forceinline__ void min_ratio(float &d, float dm, float &ratio) {
  ratio = d != 0.f ? -dm / d : -1.f;
  d = d != 0.f ? d : dm;
}

// The sum of a word's bytes, added to `acc`.
__device__ __forceinline__ uint32_t bytes_sum(uint32_t w, uint32_t acc) {
  return __builtin_amdgcn_udot4(w, 0x01010101u, acc, false);
}

// Of 0 .. most, the nearest to ratio mn / sc (0 where that is no number): where the
// block's zero lies, in units of the type's steps for it.
__device__ __forceinline__ float centre_of(float ratio, uint32_t mn, uint32_t sc, float most) {
  return fminf(fmaxf(rintf(ratio * (float)mn * __builtin_amdgcn_rcpf((float)sc)), 0.f), most);
}

// Q4_K, 144 bytes: d | dmin | scales[12] | qs[128]. Piece 0: the header; pieces
// 1 + 2 c + m: qs of 64-weight chunk c, bytes 16 m .. (piece 9 is the next
// block's and not read).
template <> struct SxtW<Q4_K> {
  static constexpr uint32_t NI = 5, UNITS = 1, BB = 144;
  static constexpr bool REM = false;
  uint32_t q[16], sc[2], mi[2];
  float d, ratio, mid;
  __device__ static void fetch(rsrc_t src, const uint8_t *reg, uint32_t voff, uint32_t bo, int, uint32_t h) {
#pragma unroll
    for (uint32_t i = 0; i < NI; ++i) dma16(src, reg + 1024u * i, voff + 16u * h, bo + 32u * i);
  }
  __device__ void take(const uint8_t *reg, int, uint32_t j, uint32_t h, uint32_t) {
    const u32x4 hd = *(const u32x4 *)(reg + 16u * j);
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const uint64_t v = lds64(reg + 512u * (p + 1) + 16u * j + 8u * h);
      q[2 * p] = (uint32_t)v;
      q[2 * p + 1] = (uint32_t)(v >> 32);
    }
    d = h2f(hd.x & 0xFFFFu);
    const uint32_t keep = d != 0.f ? 0x3F3F3F3Fu : 0u;
    sc[0] = hd.y & keep;
    mi[0] = hd.z & 0x3F3F3F3Fu;
    sc[1] = ((hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u)) & keep;
    mi[1] = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
    min_ratio(d, 32.f * h2f(hd.x >> 16), ratio);  // group sums are stored divided by 32
    mid = 4.f * centre_of(-0.0078125f * ratio, bytes_sum(mi[0], bytes_sum(mi[1], 0u)),
                          bytes_sum(sc[0], bytes_sum(sc[1], 0u)), 3.f);
  }
  // u = sc (q - c), from the nibble in a byte's high half: (1024 + 16 q) sc / 16 - (64 + c) sc, c 0, 4, 8 or 12
  // (multiples of 4: (64 + c) sc, up to 4788, is exact in fp16)
  __device__ half8 step(int s, uint32_t, const uint8_t *) const {
    const int c = s >> 2, nib = (s >> 1) & 1, m = s & 1;
    const uint32_t w0 = q[4 * c + 2 * m], w1 = q[4 * c + 2 * m + 1];
    return dec_centred((nib ? w0 : w0 << 4) & 0xF0F0F0F0u, (nib ? w1 : w1 << 4) & 0xF0F0F0F0u,
                       byte_of(sc, (uint32_t)s >> 1), 0.0625f, -64.f - mid);
  }
  // 8 minima and 8 scales: one instruction takes the sums' hi parts in k 0..7, lo in 8..15
  static constexpr uint32_t MSTEP = 1;
  __device__ half8 mins(uint32_t) const { return dec_plain(mi[0], mi[1]); }
  __device__ half8 centre(uint32_t) const { return dec_plain(sc[0], sc[1]) * (_Float16)(32.f * mid); }
};

// Q2_K, 84 bytes: scales[16] | qs[64] | d | dmin. Pieces 0: scales, 1 + 2 n + m:
// qs of the half n, bytes 16 m .., 5: d and dmin.
template <> struct SxtW<Q2_K> {
  static constexpr uint32_t NI = 3, UNITS = 1, BB = 84;
  static constexpr bool REM = false;
  uint32_t q[8], sc[4];
  float d, ratio, mid;
  __device__ static void fetch(rsrc_t src, const uint8_t *reg, uint32_t voff, uint32_t bo, int, uint32_t h) {
#pragma unroll
    for (uint32_t i = 0; i < NI; ++i) dma16(src, reg + 1024u * i, voff + 16u * h, bo + 32u * i);
  }
  __device__ void take(const uint8_t *reg, int, uint32_t j, uint32_t h, uint32_t) {
    const u32x4 s = *(const u32x4 *)(reg + 16u * j);
    const uint32_t w = lds32(reg + 512u * 5u + 16u * j);
    d = h2f(w & 0xFFFFu);
    const uint32_t kp = d != 0.f ? 0xFFFFFFFFu : 0xF0F0F0F0u;
    sc[0] = s.x & kp; sc[1] = s.y & kp; sc[2] = s.z & kp; sc[3] = s.w & kp;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint64_t v = lds64(reg + 512u * (p + 1) + 16u * j + 8u * h);
      q[2 * p] = (uint32_t)v;
      q[2 * p + 1] = (uint32_t)(v >> 32);
    }
    min_ratio(d, 16.f * h2f(w >> 16), ratio);  // group sums are stored divided by 16
    uint32_t m = 0u, t = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m = bytes_sum((sc[i] >> 4) & 0x0F0F0F0Fu, m);
      t = bytes_sum(sc[i] & 0x0F0F0F0Fu, t);
    }
    mid = 0.5f * centre_of(-0.125f * ratio, m, t, 6.f);
  }
  // u = sc (q - c), from the 2 bits at a byte's top: (1024 + 64 q) sc / 64 - (16 + c) sc, c 0, 0.5 .. 3
  __device__ half8 step(int s, uint32_t, const uint8_t *) const {
    const int n = s >> 3, g = (s >> 1) & 3, m = s & 1;
    return dec_centred((q[4 * n + 2 * m] << (6 - 2 * g)) & 0xC0C0C0C0u,
                       (q[4 * n + 2 * m + 1] << (6 - 2 * g)) & 0xC0C0C0C0u, byte_of(sc, (uint32_t)s) & 15u, 0.015625f,
                       -16.f - mid);
  }
  static constexpr uint32_t MSTEP = 2;   // 16 minima: lo, then hi
  __device__ half8 mins(uint32_t h) const {
    const uint32_t w0 = h ? sc[2] : sc[0], w1 = h ? sc[3] : sc[1];
    return dec_plain((w0 >> 4) & 0x0F0F0F0Fu, (w1 >> 4) & 0x0F0F0F0Fu);
  }
  __device__ half8 centre(uint32_t h) const {
    return dec_plain((h ? sc[2] : sc[0]) & 0x0F0F0F0Fu, (h ? sc[3] : sc[1]) & 0x0F0F0F0Fu) * (_Float16)(16.f * mid);
  }
};

// IQ2_XXS, 66 bytes: d | 8 x (4 grid indices, 4 sign fields and a scale), from
// the 4-byte floor of the block's first byte (`a`: 0 or 2 bytes before it). A
// lane keeps, per step, its grid index and sign field, and the scales. The grid
// (256 x 8 bytes) is in LDS; the sign bits come from the field and its parity
// by shifts.
template <> struct SxtW<IQ2_XXS> {
  static constexpr uint32_t NI = 3, UNITS = 1, BB = 66;
  static constexpr bool REM = false;
  uint32_t g[8], sc;   // g[i]: steps 2 i and 2 i + 1, 16 bits each: index | field << 8
  float d, ratio;
  __device__ static void fetch(rsrc_t src, const uint8_t *reg, uint32_t voff, uint32_t bo, int, uint32_t h) {
    const uint32_t v = ((voff + bo) & ~3u) + 16u * h;
#pragma unroll
    for (uint32_t i = 0; i < NI; ++i) dma16(src, reg + 1024u * i, v, 32u * i);
  }
  __device__ void take(const uint8_t *reg, int, uint32_t j, uint32_t h, uint32_t a) {
    uint32_t w[20];
#pragma unroll
    for (int p = 0; p < 5; ++p) {
      const u32x4 v = *(const u32x4 *)(reg + 512u * p + 16u * j);
      w[4 * p] = v.x; w[4 * p + 1] = v.y; w[4 * p + 2] = v.z; w[4 * p + 3] = v.w;
    }
    const uint32_t sel = a ? 0x07060504u : 0x05040302u;
    sc = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t a0 = __builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], sel) >> (8u * h);
      const uint32_t a1 = __builtin_amdgcn_perm(w[2 * i + 2], w[2 * i + 1], sel);
      sc |= (a1 >> 28) << (4 * i);
      g[i] = (a0 & 0x00FF00FFu) | (__builtin_amdgcn_ubfe(a1, 7u * h, 7u) << 8) |
             (__builtin_amdgcn_ubfe(a1, 14u + 7u * h, 7u) << 24);
    }
    d = 0.125f * h2f(a ? (w[0] >> 16) : (w[0] & 0xFFFFu));
    ratio = 0.f;
  }
  __device__ half8 step(int s, uint32_t, const uint8_t *tab) const {
    const int b = 16 * (s & 1);
    const uint64_t e = *(const uint64_t *)(tab + 8u * __builtin_amdgcn_ubfe(g[s >> 1], b, 8));
    const uint32_t f = __builtin_amdgcn_ubfe(g[s >> 1], b + 8, 7);
    const uint32_t sg = f | ((uint32_t)__builtin_popcount(f) << 7);   // bits 0..7; the eighth makes the parity even
    const half8 v = dec_scaled((uint32_t)e, (uint32_t)(e >> 32), 2u * __builtin_amdgcn_ubfe(sc, 4 * (s >> 1), 4) + 1u);
    u32x4 o = __builtin_bit_cast(u32x4, v);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // sign bits 2 i and 2 i + 1 to bits 15 and 31 (the values are not negative)
      const uint32_t m = (sg << (15 - 2 * i)) | (sg << (30 - 2 * i));
      o[i] |= m & 0x80008000u;
    }
    return __builtin_bit_cast(half8, o);
  }
  __device__ half8 mins(uint32_t) const { return half8{0, 0, 0, 0, 0, 0, 0, 0}; }
};

// Q6_K, 210 bytes: ql[128] | qh[64] | scales[16] (int8) | d, half a block (128
// weights) per unit n, from the 4-byte floor of the block's first byte. Pieces
// 0..4: ql bytes 64 n .. + 79, 5..7: qh bytes 128 + 32 n .. + 47, 8..9: scales
// and d (bytes 192 .. 223; each run one piece longer than its bytes where the
// floor moves it by 2).
template <> struct SxtW<Q6_K> {
  static constexpr uint32_t NI = 5, UNITS = 2, BB = 210;
  static constexpr bool REM = true;
  uint32_t ql[8], qh[4], sc[2];
  float d, ratio;
  __device__ static void fetch(rsrc_t src, const uint8_t *reg, uint32_t voff, uint32_t bo, int un, uint32_t h) {
    const uint32_t v = (voff + bo) & ~3u, n = (uint32_t)un, vh = v + 16u * h;
    dma16(src, reg, vh, 64u * n);
    dma16(src, reg + 1024u, vh, 64u * n + 32u);
    dma16(src, reg + 2048u, v + (h ? 128u + 32u * n : 64u + 64u * n), 0u);
    dma16(src, reg + 3072u, vh, 144u + 32u * n);
    dma16(src, reg + 4096u, vh, 192u);
  }
  __device__ void take(const uint8_t *reg, int un, uint32_t j, uint32_t h, uint32_t a) {
    const uint8_t *p0 = reg + 16u * j + 8u * h;             // the lane's 8 bytes of a piece
    const uint8_t *p1 = reg + 16u * j + (h ? 512u : 8u);    // and the dword after them
    auto get = [&](int p, uint32_t &o0, uint32_t &o1) {
      const uint64_t w = lds64(p0 + 512 * p);
      const uint32_t w2 = lds32(p1 + 512 * p);
      o0 = __builtin_amdgcn_alignbyte((uint32_t)(w >> 32), (uint32_t)w, a);
      o1 = __builtin_amdgcn_alignbyte(w2, (uint32_t)(w >> 32), a);
    };
#pragma unroll
    for (int p = 0; p < 4; ++p) get(p, ql[2 * p], ql[2 * p + 1]);
#pragma unroll
    for (int p = 0; p < 2; ++p) get(5 + p, qh[2 * p], qh[2 * p + 1]);
    const uint8_t *ps = reg + 512u * 8u + 16u * j;
    const uint64_t s01 = lds64(ps + 8 * un);
    const uint32_t s2 = lds32(un ? ps + 512 : ps + 8), w = lds32(ps + 512);
    sc[0] = __builtin_amdgcn_alignbyte((uint32_t)(s01 >> 32), (uint32_t)s01, a);
    sc[1] = __builtin_amdgcn_alignbyte(s2, (uint32_t)(s01 >> 32), a);
    d = h2f(a ? (w >> 16) : (w & 0xFFFFu));
    ratio = 0.f;
  }
  // step s of the unit (0..7): v = fp16(sc (q - 32)) and what it is off by
  __device__ half8 step2(int s, half8 &rem) const {
    const int g = s >> 1, m = s & 1, p = 2 * (g & 1) + m, ls = 4 * (g >> 1), hs = 2 * g;
    const uint32_t u0 = ((ql[2 * p] >> ls) & 0x0F0F0F0Fu) | (((qh[2 * m] >> hs) & 0x03030303u) << 4);
    const uint32_t u1 = ((ql[2 * p + 1] >> ls) & 0x0F0F0F0Fu) | (((qh[2 * m + 1] >> hs) & 0x03030303u) << 4);
    const half2v o2 = {(_Float16)-1056.f, (_Float16)-1056.f};   // 1024 + q - 1056 = q - 32
    const _Float16 c = (_Float16)(float)(int8_t)byte_of(sc, (uint32_t)s);
    const half2v c2 = {c, c};
    const half2v e[4] = {h1024_lo(u0) + o2, h1024_hi(u0) + o2, h1024_lo(u1) + o2, h1024_hi(u1) + o2};
    half8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const half2v t = e[i] * c2, r = __builtin_elementwise_fma(e[i], c2, -t);
      v[2 * i] = t.x; v[2 * i + 1] = t.y;
      rem[2 * i] = r.x; rem[2 * i + 1] = r.y;
    }
    return v;
  }
  __device__ half8 mins(uint32_t) const { return half8{0, 0, 0, 0, 0, 0, 0, 0}; }
};

// s_waitcnt vmcnt(N) lgkmcnt(0): the loads past the N youngest are in, and
// every LDS read of this wave has returned.
template <uint32_t N>
__device__ __forceinline__ void wait_vm_lds() {
  static_assert(N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((int)((N & 15u) | ((N >> 4) << 14) | 0x0070u));
}

constexpr uint32_t kTokTile = 64;    // tokens per workgroup: 4 tiles of 16 of the prepared x
constexpr uint32_t kBand = 4;        // token tiles of a band of the tile order
constexpr uint32_t kSxtLorBlocks = 7;    // Q6_K: blocks of k up to which lo times r is taken too

template <int TYPE>
struct SxtLds {
  static constexpr uint32_t XG = 2u * 4u * 4096u;                   // 4 steps of 64 tokens, for each k slice
  static constexpr uint32_t WR = SxtW<TYPE>::NI * 1024u;            // raw weights of 32 rows
  static constexpr uint32_t TAB = TYPE == IQ2_XXS ? 2048u : 0u;
  static constexpr uint32_t X0 = TAB, W0 = X0 + 2u * XG, M0 = W0 + 8u * WR;
  static constexpr uint32_t P0 = M0 + (sx_mins<TYPE>() ? 8192u : 0u);   // group sums of a block, for each k slice
  static constexpr uint32_t LOOP = P0 + 1024u;                      // block scales: 2 blocks x 2 slices x 64 tokens
  static constexpr uint32_t RED = 8u * 4096u + 16u;                 // the waves' sums handed over
  static constexpr uint32_t BYTES = LOOP > RED ? LOOP : RED;
  static_assert(BYTES <= 160u * 1024u, "LDS");
};

__device__ __forceinline__ float16v mma(half8 a, half8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// LOR: lo times r as well (Q6_K)
template <int TYPE, bool LOR>
__global__ __launch_bounds__(512) void k_sxt(WeightView wv, const uint8_t *__restrict__ xa,
                                             const float *__restrict__ xp, float *__restrict__ y, uint32_t tokens,
                                             uint32_t xa_bytes, uint32_t xp_bytes, uint32_t row_tiles,
                                             uint32_t tok_tiles, uint32_t ksl, float *__restrict__ part,
                                             uint32_t *__restrict__ cnt) {
  using W = SxtW<TYPE>;
  using L = SxtLds<TYPE>;
  constexpr bool MINS = sx_mins<TYPE>();
  constexpr bool HALF = MINS || W::REM;          // a block's hi parts in two sums of 8 steps
  constexpr uint32_t NS = sx_slots<TYPE>();
  static_assert(!LOR || W::REM, "r");
  constexpr uint32_t SU = 16u / W::UNITS;        // steps of a unit
  constexpr uint32_t WI = W::NI;                 // a wave's loads of a unit's weights
  constexpr uint32_t XI = 4u;                    // and of a group's x
  __shared__ __align__(16) uint8_t lds[L::BYTES];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, j = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), rg = wave & 3u, ks = wave >> 2;

  // Workgroups of one XCD (blockIdx % 8) take a contiguous run of (k slice, tile)
  // pairs, in bands of 4 token tiles, token tiles fastest: the 32 tiles an XCD has
  // at a time are 4 x 8, and share x and weights through its L2. Over all token
  // tiles at once every CU read x of its own (us, Q4_K 8192 x 2048 at 2048 tokens 219
  // / bands of 4 193 / of 8 194, IQ2_XXS 210 / 193 / 192, Q4_K 4096 x 4096 at 1500 145 /
  // 141 / 139, 8192 x 2048 at 700 74.3 / 74.4 / 75.4, at 512 53.7 all).
  const uint32_t ntiles = row_tiles * tok_tiles, nwg = ntiles * ksl;
  uint32_t u = blockIdx.x;
  if (nwg % 8u == 0u) u = (blockIdx.x % 8u) * (nwg / 8u) + blockIdx.x / 8u;
  const uint32_t z = u / ntiles, lin = u - z * ntiles;
  const uint32_t band = lin / (kBand * row_tiles), bi = lin - band * kBand * row_tiles;
  const uint32_t bw = min(kBand, tok_tiles - kBand * band);   // the last band's may be fewer
  const uint32_t tt0 = kBand * band + bi % bw, r0 = (bi / bw) * 128u + 32u * rg;
  const uint32_t rows = wv.rows, nb = wv.k / 256u;
  const uint32_t bl = z * nb / ksl, bh = (z + 1u) * nb / ksl, iters = (bh - bl + 1u) / 2u;

  if constexpr (TYPE == IQ2_XXS) {
    if (tid < 256u) *(uint64_t *)(lds + 8u * tid) = c_grid_sxt[tid];
  }

  const rsrc_t wsrc = make_rsrc(wv.w, wv.w_bytes), xsrc = make_rsrc(xa, xa_bytes), psrc = make_rsrc(xp, xp_bytes);
  const uint32_t wrow = min(r0 + j, rows - 1u) * (uint32_t)wv.row_bytes;
  uint8_t *const wreg = lds + L::W0 + wave * L::WR;
  const uint32_t pvoff = ((4u * tt0 + (lane >> 4)) * nb * 16u + (lane & 15u)) * 4u;
  const uint32_t xtile = (4u * tt0 + (wave & 3u)) * nb;

  // the block of slice sl in iteration it (loads past the end repeat the last block)
  auto blk = [&](uint32_t it, uint32_t sl) { return min(bl + 2u * it + sl, bh - 1u); };
  auto fetch_w = [&](uint32_t it, int un) { W::fetch(wsrc, wreg, wrow, blk(it, ks) * W::BB, un, h); };
  // x of group g (4 steps) of iteration it: 1 KB chunk c = wave + 8 i is
  // 16-token tile c % 4 of step c / 4 % 4 of slice c / 16
  auto fetch_x = [&](uint32_t it, uint32_t g) {
#pragma unroll
    for (uint32_t i = 0; i < XI; ++i) {
      const uint32_t s = ((wave >> 2) + 2u * i) & 3u;
      dma16(xsrc, lds + L::X0 + (g & 1u) * L::XG + (wave + 8u * i) * 1024u, 16u * lane,
            ((xtile + blk(it, i >> 1)) * NS + 4u * g + s) * 1024u);
    }
  };
  // the group sums (one 1 KB chunk per wave) and block scales of iteration it
  auto fetch_m = [&](uint32_t it) {
    if constexpr (MINS)
      dma16(xsrc, lds + L::M0 + wave * 1024u, 16u * lane, ((xtile + blk(it, wave >> 2)) * NS + 16u) * 1024u);
    dma4(psrc, lds + L::P0 + (it & 1u) * 512u + ks * 256u, pvoff, blk(it, ks) * 64u);
  };
  // the lane's fragment rows: token j of a tile of 32 = row j % 16 of 16-token tile j / 16
  const uint8_t *const xl = lds + L::X0 + ks * 16384u + (j >> 4) * 1024u + 16u * (32u * h + (j & 15u));

  // by token tile of 32. D: a block's sums of the hi parts (HALF: of its second
  // half, E holding the first's), D2: of the lo parts and of the products with r;
  // acc: the folded sums of a run of blocks, total: of the runs before it
  float16v total[2], acc[2], D[2], D2[2], E[HALF ? 2 : 1];
#pragma unroll
  for (int a = 0; a < 2; ++a) total[a] = acc[a] = float16v{};
  auto end_run = [&]() {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int v = 0; v < 16; ++v) total[a][v] += acc[a][v];
      acc[a] = float16v{};
    }
  };

  W w;
  auto take_w = [&](uint32_t it, int un) {
    w.take(wreg, un, j, h, (wrow + blk(it, ks) * W::BB) & 2u);
    // every read of the region has returned before the next loads into it go out
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  half8 A[2][2];   // [part][tile]: the present step's until its instructions are issued, then the next one's
  auto read_a = [&](int q, uint32_t g, uint32_t i) {
    const uint8_t *p = xl + (g & 1u) * L::XG + i * 4096u + 256 * q;
#pragma unroll
    for (int a = 0; a < 2; ++a) A[q][a] = *(const half8 *)(p + 2048 * a);
    __asm__ volatile("" ::: "memory");
  };
  half8 B[2], R[2];
  auto decode = [&](uint32_t set, uint32_t s) {
    if constexpr (W::REM) B[set] = w.step2((int)(s % SU), R[set]);
    else B[set] = w.step((int)s, h, lds);
  };
  auto low = [&](uint32_t set) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      D2[a] = mma(A[1][a], B[set], D2[a]);
      if constexpr (LOR) D2[a] = mma(A[1][a], R[set], D2[a]);
    }
  };
  auto high = [&](uint32_t set) {
#pragma unroll
    for (int a = 0; a < 2; ++a) D[a] = mma(A[0][a], B[set], D[a]);
    if constexpr (W::REM) {
#pragma unroll
      for (int a = 0; a < 2; ++a) D2[a] = mma(A[0][a], R[set], D2[a]);
    }
  };
  // D at the start of a block: the minima's sums, scaled, and the centre's
  float dcur;
  auto open = [&]() {
#pragma unroll
    for (int a = 0; a < 2; ++a) D[a] = D2[a] = float16v{};
    if constexpr (MINS) {
      const uint8_t *ml =
          lds + L::M0 + ks * 4096u + (j >> 4) * 1024u + 16u * ((W::MSTEP == 1u ? 16u : 32u) * h + (j & 15u));
      half8 ms[2][W::MSTEP];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (uint32_t q = 0; q < W::MSTEP; ++q) ms[a][q] = *(const half8 *)(ml + 2048 * a + 256u * q);
      const half8 mb = w.mins(h), cb = w.centre(h);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int q = (int)W::MSTEP - 1; q >= 0; --q) D[a] = mma(ms[a][q], mb, D[a]);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int v = 0; v < 16; ++v) D[a][v] *= w.ratio;
#pragma unroll
        for (int q = (int)W::MSTEP - 1; q >= 0; --q) D[a] = mma(ms[a][q], cb, D[a]);
      }
    }
    dcur = w.d;
  };

  // prologue: the first unit's weights, the first block's sums and scales, x of
  // the first two groups
  fetch_w(0u, 0);
  fetch_m(0u);
  fetch_x(0u, 0u);
  wait_vm<0>();
  __syncthreads();
  fetch_x(0u, 1u);
  take_w(0u, 0);
  fetch_w(W::UNITS == 1u ? 1u : 0u, W::UNITS == 1u ? 0 : 1);
  read_a(1, 0u, 0u);
  read_a(0, 0u, 0u);
  decode(0u, 0u);

  // more than 12 blocks in runs of a quarter of them: as many partial sums as the
  // waves of k_sx make (one run of 28 blocks: 1.1 of k_sx's error for sums of one
  // sign; the runs cost 1-2% of the time at 4 to 8 blocks, where one is as exact)
  const uint32_t run = iters > 12u ? (iters + 3u) / 4u : iters;
  for (uint32_t it = 0; it < iters;) {
    for (const uint32_t end = min(it + run, iters); it < end; ++it) {
      open();
#pragma unroll
      for (uint32_t s = 0; s < 16u; ++s) {
        const uint32_t cur = s & 1u, nxt = cur ^ 1u, g = s >> 2, gn = (g + ((s & 3u) == 3u)) & 3u, sn = (s + 1u) & 3u;
        if constexpr (HALF)
          if (s == 8u) {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              E[a] = D[a];
              D[a] = float16v{};
            }
          }
        // lo parts; at a group's end, between the two, the next group's x is in
        // LDS once every wave's own loads of it are (a group ago; the weights of
        // the next unit went out after them), and the present group's buffer is
        // free once every wave has read it
        low(cur);
        if ((s & 3u) == 3u) {
          __builtin_amdgcn_sched_barrier(0);
          if (g % (W::UNITS == 1u ? 4u : 2u) == 0u) wait_vm_lds<WI>();
          else wait_vm_lds<0>();
          __builtin_amdgcn_s_barrier();
          __asm__ volatile("" ::: "memory");
          if (g == 2u) fetch_m(it + 1u);
          fetch_x(g < 2u ? it : it + 1u, (g + 2u) & 3u);
        }
        read_a(1, gn, sn);
        if ((s + 1u) % SU == 0u) {
          // the next unit: its weights into registers, and the loads of the one after
          const uint32_t ni = s == 15u ? it + 1u : it;
          const int un = s == 15u ? 0 : 1;
          take_w(ni, un);
          fetch_w(un + 1 == (int)W::UNITS ? ni + 1u : ni, un + 1 == (int)W::UNITS ? 0 : un + 1);
        }
        // hi parts, while the next step's weights are decoded
        decode(nxt, (s + 1u) & 15u);
        high(cur);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        }
        read_a(0, gn, sn);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the fold
      if (bl + 2u * it + ks < bh) {
        const uint8_t *pp = lds + L::P0 + (it & 1u) * 512u + ks * 256u + 16u * h;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4 p = *(const float4 *)(pp + 128 * a + 32 * g);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              float t = D[a][4 * g + v] + D2[a][4 * g + v];
              if constexpr (HALF) t += E[a][4 * g + v];
              acc[a][4 * g + v] =
                  __builtin_fmaf(t * dcur, v == 0 ? p.x : v == 1 ? p.y : v == 2 ? p.z : p.w, acc[a][4 * g + v]);
            }
          }
      }
    }
    end_run();
  }
  wait_vm<0>();
  __syncthreads();

  // the two k slices' sums, slice 0 + slice 1: a wave writes token tile ks of its
  // 32 rows and hands the other over in LDS
  float *const red = (float *)lds;
  float16v sum;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    sum[v] = ks ? total[1][v] : total[0][v];
    red[(wave * 16u + v) * 64u + lane] = ks ? total[0][v] : total[1][v];
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < 16; ++v) sum[v] += red[((wave ^ 4u) * 16u + v) * 64u + lane];

  if (ksl > 1u) {
    // k slices over workgroups, as in eff_gemm_sx.hip: the last of the tile's
    // ksl workgroups to arrive adds the slices, two by two, the pairs in order (all in
    // a row, sums of one sign over 6 slices came to 1.06 of k_sx's error)
    constexpr int kSc1 = 16;   // cache policy bit 4: sc1
    constexpr uint32_t NE = kTokTile * 128u;
    uint32_t *const arrived = (uint32_t *)(lds + L::BYTES - 16u);
    const rsrc_t prs = make_rsrc(part + (uint64_t)lin * ksl * NE, (uint64_t)ksl * NE * 4u);
    auto off = [&](uint32_t zz, uint32_t v4) {
      return (int)(zz * (NE * 4u) + ((wave * 4u + v4) * 64u + lane) * 16u);
    };
#pragma unroll
    for (uint32_t v = 0; v < 4u; ++v) {
      const u32x4 o = {__float_as_uint(sum[4 * v]), __float_as_uint(sum[4 * v + 1]), __float_as_uint(sum[4 * v + 2]),
                       __float_as_uint(sum[4 * v + 3])};
      __builtin_amdgcn_raw_buffer_store_b128(o, prs, off(z, v), 0, kSc1);
    }
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // every wave's sums are stored
    if (tid == 0u) *arrived = __hip_atomic_fetch_add(cnt + lin, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != ksl - 1u) return;
    if (tid == 0u) __hip_atomic_store(cnt + lin, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t zz = 0; zz < ksl; zz += 2u) {
      const bool two = zz + 1u < ksl;
#pragma unroll
      for (uint32_t v = 0; v < 4u; ++v) {
        const u32x4 o = __builtin_amdgcn_raw_buffer_load_b128(prs, off(zz, v), 0, kSc1);
        const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(prs, off(two ? zz + 1u : zz, v), 0, kSc1);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float t = two ? __uint_as_float(o[c]) + __uint_as_float(q[c]) : __uint_as_float(o[c]);
          sum[4 * v + c] = zz ? sum[4 * v + c] + t : t;
        }
      }
    }
  }
  // written through L2 (us, plain / nontemporal / written through, and with the next
  // layer's product, which reads y: Q4_K 8192 x 2048 at 512 tokens 50.6 / 49.0 / 49.1
  // and 104.3 / 104.0 / 102.7, Q6_K 2048 x 8192 at 300 53.5 / 52.0 / 51.4 and 93.5 /
  // 91.6 / 91.0)
  const uint32_t row = r0 + j;
  if (row >= rows) return;
#pragma unroll
  for (uint32_t v = 0; v < 16u; ++v) {
    const uint32_t tok = kTokTile * tt0 + 32u * ks + 8u * (v >> 2) + 4u * h + (v & 3u);
    if (tok < tokens) store_through(y + (uint64_t)tok * rows + row, sum[v]);
  }
}

struct SxtPlan {
  uint32_t row_tiles, tok_tiles, ksl;
};

SxtPlan sxt_plan(const WeightView &wv, uint32_t tokens, uint32_t ksl) {
  return {(wv.rows + 127u) / 128u, (tokens + kTokTile - 1u) / kTokTile, (uint32_t)max(1u, min(ksl, wv.k / 256u))};
}

template <int TYPE>
hipError_t sxt_go(const WeightView &wv, const uint8_t *xa, const float *xp, uint32_t tiles, float *y,
                  uint32_t tokens, const SxtPlan &p, void *sk, hipStream_t s) {
  const uint64_t nb = wv.k / 256u, xb = (uint64_t)tiles * nb * sx_slots<TYPE>() * 1024u;
  if (tiles < 4u * p.tok_tiles || xb >= (1ull << 32)) return hipErrorInvalidValue;
  if (p.ksl > 1u && (!sk || (uint64_t)p.row_tiles * p.tok_tiles > kSliceCntBytes / 4u)) return hipErrorInvalidValue;
  uint32_t *cnt = (uint32_t *)sk;
  float *part = sk ? (float *)((uint8_t *)sk + kSliceCntBytes) : nullptr;
  constexpr bool REM = SxtW<TYPE>::REM;
  auto *const kernel = REM && nb <= kSxtLorBlocks ? k_sxt<TYPE, REM> : k_sxt<TYPE, false>;
  hipLaunchKernelGGL(kernel, dim3(p.row_tiles * p.tok_tiles * p.ksl), dim3(512), 0, s, wv, xa, xp, y, tokens,
                     (uint32_t)xb, (uint32_t)(tiles * nb * 64u), p.row_tiles, p.tok_tiles, p.ksl, part, cnt);
  return hipGetLastError();
}

}  // namespace

size_t sxt_sk_bytes(const WeightView &wv, uint32_t tokens, uint32_t ksl) {
  const SxtPlan p = sxt_plan(wv, tokens, ksl);
  if (p.ksl < 2u) return 0;
  return kSliceCntBytes + (size_t)p.row_tiles * p.tok_tiles * p.ksl * (kTokTile * 128u * 4u);
}

hipError_t launch_sxt(const WeightView &wv, const void *xa, const void *xp, uint32_t tiles, float *y,
                      uint32_t tokens, uint32_t ksl, void *sk, hipStream_t s) {
  const SxtPlan p = sxt_plan(wv, tokens, ksl);
  const uint8_t *a = (const uint8_t *)xa;
  const float *b = (const float *)xp;
  switch (wv.type) {
    case Q4_K: return sxt_go<Q4_K>(wv, a, b, tiles, y, tokens, p, sk, s);
    case Q6_K: return sxt_go<Q6_K>(wv, a, b, tiles, y, tokens, p, sk, s);
    case Q2_K: return sxt_go<Q2_K>(wv, a, b, tiles, y, tokens, p, sk, s);
    case IQ2_XXS: return sxt_go<IQ2_XXS>(wv, a, b, tiles, y, tokens, p, sk, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace eff
