// Fused dequant-GEMV on raw GGUF rows for 2 to 16 tokens, on gfx950's matrix
// cores (nsx_fused_gemv; the reference's compute/triton_kernels.py:199-228
// fuses one token).
//
// y = x . W^T with every weight code exact in bf16 and every activation as the
// sum of three bf16 terms of a power-of-two-scaled copy: its 24 bits, whatever
// the token's other activations are (gm_split says down to where), so the
// products are those of fp32 values, and the matrix cores' sums are fp32.
// v_mfma_f32_16x16x32_bf16 with A = 16 rows of terms x 32 elements and B = 32
// elements x 16 weight rows. The 16 rows of A are
//   up to 5 tokens:  row j = term j / 5 of token j % 5, one instruction;
//   up to 8:  row j = term j / 8 of token j % 8, then a second instruction
//     whose rows j < 8 are term 2;
//   up to 16: row j = token j, one instruction per term.
// A lane holds one weight row's codes and the same row's results, so the
// block scales multiply its own registers, without a shuffle.
//
// A workgroup is 8 or 16 waves; each takes its part of K and keeps its terms in
// registers for every row it meets (a small kernel lays them out in the
// caller's workspace: no LDS or cache traffic for activations in the loop). Per 16-row tile a wave reads its part of the
// rows with 16-byte loads, coalesced along the rows, parks them in LDS (a
// private buffer, so that a lane can pick up its codes at any byte offset),
// requests the next tile's, and multiplies; the partial sums meet in LDS
// in a fixed order, one barrier per tile. Where K exceeds what the waves hold,
// K is taken in passes over groups of GM_GROUP tiles whose sums wait in LDS.
//
// Bound: the weight bytes, then the decode's VALU instructions (about 20 per 8 codes
// of a lane). Measured, 200000 x 2880, one call: Q8_0 at 8 tokens 146 us (4.2 TB/s) against 1150
// for the VALU kernel, which decodes a weight per 4 tokens; MXFP4 at 5 tokens 81 / 622; Q4_0 95 /
// 626; Q4_K 95 / 645; Q6_K 172 / 494. (Terms and codes in f16, whose packed arithmetic decodes with fewer
// instructions: 142, 81, 82, 97, 155, but a token's small values lost bits beside a large one.)
#include "gemv_mm.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int GM_ROWS = 16;    // weight rows of a tile
constexpr int GM_GROUP = 16;   // tiles whose sums wait in LDS between passes over K
constexpr int GM_PS = 20;      // floats between the A rows of a partial tile (conflict-free writes)
constexpr int GM_MAXT = 16;

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));  // four bf16 (the 16-element product's operands)

// A format's K unit (the smallest part of a row with scales of its own): elements, bytes.
template <int FMT> struct Unit { static constexpr int E = 32, B = FMT == NSX_Q8_0 ? 34 : FMT == NSX_Q4_0 ? 18 : 17; };
template <> struct Unit<NSX_Q4_K> { static constexpr int E = 256, B = 144; };
template <> struct Unit<NSX_Q6_K> { static constexpr int E = 256, B = 210; };

// Waves of a workgroup: 16 where a sixteenth of K leaves each its 128 registers without spilling, else 8 with 256
// (200000 x 2880: Q4_0 at 5 tokens 95 us against 104 with 8 waves, at 8 tokens 96 / 103, but at 16 tokens 133 / 111;
// MXFP4 65536 x 4096 at 5 tokens 40 / 50; Q8_0 120 / 142, at 8 tokens 167 / 146; Q4_K and Q6_K blocks of 256 spill).
template <int FMT>
constexpr int gm_waves(int nm) { return Unit<FMT>::E == 32 && nm <= (FMT == NSX_Q8_0 ? 1 : 2) ? 16 : 8; }
// Elements a wave holds terms for, in 32s: 4 registers per 32 elements and instruction, what the staged pieces leave of
// the lane's registers (Q8_0 at 8 tokens, 65536 x 4096: 16 of them, spilling, 100 us, two passes of 8 75 us).
template <int FMT>
constexpr int gm_max_e32(int nm) {
  if (gm_waves<FMT>(nm) == 16) return nm == 1 && FMT != NSX_Q8_0 ? 8 : 6;
  if (FMT == NSX_Q8_0) return nm == 2 ? 12 : 8;
  if (FMT == NSX_Q6_K) return nm == 1 ? 16 : 8;
  return nm == 3 ? (FMT == NSX_Q4_K ? 8 : 12) : 16;
}

// 16-byte pieces of one row's part of a tile, which are the row's stride in LDS: not a multiple of 4, so that the 16
// rows' reads spread over the banks.
__host__ __device__ constexpr int gm_pieces(int bytes) {
  const int n = (bytes + 3 + 15) / 16;
  return n % 4 ? n : n + 1;
}

// A lane's weight row in LDS, whose first byte may sit at any offset modulo 4. Whole code words are read from the
// aligned dwords around them and realigned in registers (a misaligned LDS word costs several aligned ones); c is the
// word's place past the lane group's part, a constant, so that one of four addresses and shifts serves it.
struct LdsRow {
  const uint8_t* p;      // the row
  const uint8_t* at[4];  // dword that holds byte k of the lane group's part of the row
  uint32_t sh[4];        // place of that byte in it
  __device__ __forceinline__ void set(const uint8_t* aligned, uint32_t res, uint32_t part) {
    p = aligned + res;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      at[k] = aligned + part + ((res + k) & ~3u);
      sh[k] = (res + k) & 3u;
    }
  }
  __device__ __forceinline__ uint32_t word(int c) const {
    const uint32_t* d = (const uint32_t*)(at[c & 3] + (c & ~3));
    return nsx_alignbyte(d[1], d[0], sh[c & 3]);
  }
  __device__ __forceinline__ v2u words(int c) const {
    const uint32_t* d = (const uint32_t*)(at[c & 3] + (c & ~3));
    return v2u{nsx_alignbyte(d[1], d[0], sh[c & 3]), nsx_alignbyte(d[2], d[1], sh[c & 3])};
  }
  template <typename T>
  __device__ __forceinline__ T get(int c) const {  // (gfx950 reads LDS at any byte offset)
    T v;
    __builtin_memcpy(&v, p + c, sizeof(T));
    return v;
  }
};

// Two bf16 from the halves of two fp32 whose lower halves are zero.
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
}
__device__ __forceinline__ float byte_of(uint32_t w, int i) { return (float)((w >> (8 * i)) & 0xFFu); }
__device__ __forceinline__ float sbyte_of(uint32_t w, int i) { return (float)(int8_t)(w >> (8 * i)); }
// Four bytes, unsigned or signed, as bf16.
__device__ __forceinline__ v2u bytes4(uint32_t w) {
  return v2u{pack2(byte_of(w, 0), byte_of(w, 1)), pack2(byte_of(w, 2), byte_of(w, 3))};
}
__device__ __forceinline__ v2u sbytes4(uint32_t w) {
  return v2u{pack2(sbyte_of(w, 0), sbyte_of(w, 1)), pack2(sbyte_of(w, 2), sbyte_of(w, 3))};
}
// Four bytes of 0..15 as bf16: as fp8 (e4m3) such a byte is its value / 512, subnormal or not.
__device__ __forceinline__ v2u nibbles4(uint32_t w) {
  return v2u{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.f, false)),
             __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.f, true))};
}
// Bytes 2 B and 2 B + 1 of e2m1 codes, a byte's low one first, as bf16 times 2.
template <int B>
__device__ __forceinline__ v2u fp4x4(uint32_t w) {
  return v2u{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 2.f, 2 * B)),
             __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 2.f, 2 * B + 1))};
}
// The codes above and below are taken as bytes whose low bits are zero: 2^this times the weight's.
template <int FMT> constexpr int GM_CODE_EXP = FMT == NSX_Q4_0 ? 4 : FMT == NSX_Q6_K ? 2 : 0;

template <int NM>
__device__ __forceinline__ int gm_token(int j) { return NM == 1 ? j % 5 : NM == 2 ? j % 8 : j; }

// ---------------------------------------------------------------------------
// Activation terms, laid out as the lanes of the product kernel hold them:
//   per unit and instruction m its operands, [piece][lane][16 B]: a format of 32-element units has one piece; Q4_K
//   eight (sub-blocks 0..7) and one with the sub-blocks' sums (lane group 0: elements 0..7; zero elsewhere);
//   Q6_K eight of two 16-element products each;
//   then 16 exponents: slot j's sums are 2^(its exponent) times its token's.
template <int FMT> constexpr int GM_PIECES = FMT == NSX_Q4_K ? 9 : FMT == NSX_Q6_K ? 8 : 1;
template <int FMT>
__host__ __device__ constexpr int64_t gm_terms_bytes(int64_t K, int nm) {
  return K / Unit<FMT>::E * GM_PIECES<FMT> * nm * 1024;
}

// Element (of the unit) at place v (0..7) of piece pc of lane group g.
template <int FMT>
__device__ __forceinline__ int gm_elem(int pc, int g, int v) {
  if constexpr (FMT == NSX_Q8_0) return 8 * g + v;
  else if constexpr (FMT == NSX_Q4_K) return 32 * pc + 8 * g + v;
  else if constexpr (FMT == NSX_Q4_0) return 4 * g + (v & 3) + 16 * (v >> 2);   // low nibbles, then high ones
  else if constexpr (FMT == NSX_MXFP4) return 4 * g + (v >> 1) + 16 * (v & 1);  // a byte's low and high code side by side
  else {  // Q6_K: products 2 pc and 2 pc + 1; product 4 (2 h + hl) + L holds elements 128 h + 32 L + 16 hl ..
    const int pr = 2 * pc + (v >> 2), hh = pr >> 2, L = pr & 3;
    return 128 * (hh >> 1) + 32 * L + 16 * (hh & 1) + 4 * g + (v & 3);
  }
}

// Terms 0..2 of the scaled activation v: its leading 8 bits, the next 8, the rest, each exact in bf16. The token's
// largest finite |x| goes to 2^60 .. 2^61: an activation down to 2^-160 of it keeps all its 24 bits (terms from 2^-126 on
// are normal), and the sums of a row stay within fp32's range. (One grid of f16 terms for a token would lose a bit for
// each factor of two below 2^-15 of its largest value: with that value under a zero code, what is left of the row.) An
// infinite or NaN v is its own first term.
constexpr int GM_TOP = 61;  // the largest |x| < 2^GM_TOP
__device__ __forceinline__ void gm_split(float v, uint16_t (&t)[3]) {
  auto top = [](float x) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xFFFF0000u); };
  const bool fin = fabsf(v) <= 3.4028235e38f;
  const float hi = top(v), r = fin ? v - hi : 0.f, mid = top(r), lo = r - mid;
  t[0] = (uint16_t)((__builtin_bit_cast(uint32_t, v) >> 16) | (v != v ? 0x40u : 0u));  // (a NaN stays one)
  t[1] = (uint16_t)(__builtin_bit_cast(uint32_t, mid) >> 16);
  t[2] = (uint16_t)(__builtin_bit_cast(uint32_t, lo) >> 16);
}

// Workgroup (token, part of K): the token's scale from the whole row,
// then its slots' terms of the part's units; token 0's workgroups clear the slots that hold no token.
template <int FMT, int NM>
__global__ __launch_bounds__(256) void gm_terms_kernel(const void* __restrict__ x, int dt, int K, int T,
                                                       uint8_t* __restrict__ ws) {
  constexpr int UE = Unit<FMT>::E, PC = GM_PIECES<FMT>, ROWS = UE / 8;  // 8-element runs of a unit
  __shared__ float part[4];
  const int tok = blockIdx.x, tid = threadIdx.x;
  const int64_t x0 = (int64_t)tok * K;
  float mx = 0.f;
  for (int k = tid; k < K; k += 256 * 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = nsx_load_act(x, dt, x0 + min(k + 256 * i, K - 1));
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fabsf(v[i]) <= 3.4028235e38f ? fmaxf(mx, fabsf(v[i])) : mx;
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((tid & 63) == 0) part[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  int ex = GM_TOP;
  if (mx > 0.f) (void)frexpf(mx, &ex);  // mx < 2^ex
  const int e = GM_TOP - ex;
  int32_t* exps = (int32_t*)(ws + gm_terms_bytes<FMT>(K, NM));
  auto store = [&](int slot, int m, int u, int pc, int g, const v4u& h) {
    *(v4u*)(ws + ((((int64_t)u * PC + pc) * NM + m) * 64 + 16 * g + slot) * 16) = h;
  };
  // run r of 8 elements -> piece pc = r / 4 of lane group g = r % 4 (Q4_K's sums: below)
  const int runs = K / 8, per = (runs + (int)gridDim.y - 1) / (int)gridDim.y;
  const int r1 = min(runs, per * ((int)blockIdx.y + 1));
  for (int r = per * (int)blockIdx.y + tid; r < r1; r += 256) {
    const int u = r / ROWS, pc = (r % ROWS) >> 2, g = r & 3;
    uint16_t t[8][3];
#pragma unroll
    for (int v = 0; v < 8; ++v)
      gm_split(ldexpf(nsx_load_act(x, dt, x0 + (int64_t)u * UE + gm_elem<FMT>(pc, g, v)), e), t[v]);
#pragma unroll
    for (int term = 0; term < 3; ++term) {
      v4u h;
#pragma unroll
      for (int v = 0; v < 4; ++v) h[v] = t[2 * v][term] | (uint32_t)t[2 * v + 1][term] << 16;
      if (NM == 1) store(5 * term + tok, 0, u, pc, g, h);
      else if (NM == 2) store(term == 1 ? 8 + tok : tok, term == 2 ? 1 : 0, u, pc, g, h);
      else store(tok, term, u, pc, g, h);
    }
  }
  if constexpr (FMT == NSX_Q4_K) {  // one thread per super-block of this workgroup's part
    const int all = K / UE, pu = (all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int u = pu * (int)blockIdx.y + (tid >> 3);  // 8 threads per unit, one sub-block each
    const bool on = (tid >> 3) < pu && u < all;
    float s = 0.f;
    for (int i = 0; i < 32; ++i) s += on ? ldexpf(nsx_load_act(x, dt, x0 + (int64_t)u * UE + 32 * (tid & 7) + i), e) : 0.f;
    uint16_t t[3];
    gm_split(s, t);
    if (on) {
#pragma unroll
      for (int term = 0; term < 3; ++term) {
        const int slot = NM == 1 ? 5 * term + tok : NM == 2 ? (term == 1 ? 8 + tok : tok) : tok;
        const int m = NM == 1 ? 0 : NM == 2 ? (term == 2 ? 1 : 0) : term;
        uint8_t* p = ws + ((((int64_t)u * PC + 8) * NM + m) * 64 + slot) * 16;
        *(uint16_t*)(p + 2 * (tid & 7)) = t[term];
        for (int g = 1; g < 4; ++g) *(uint16_t*)(p + 16 * 16 * g + 2 * (tid & 7)) = 0;
      }
    }
  }
  if (blockIdx.y == 0 && tid < 16 && gm_token<NM>(tid) == tok) exps[tid] = e + GM_CODE_EXP<FMT>;
  if (tok == 0) {  // slots without a token (NM 2: the second instruction has 8 more)
    const int all = K / UE * PC;
    for (int i = (int)blockIdx.y * 256 + tid; i < all * NM * 64; i += 256 * (int)gridDim.y) {
      const int slot = i & 15, m = (i >> 6) % NM;
      const bool none = gm_token<NM>(slot) >= T || (NM == 1 && slot == 15) || (NM == 2 && m == 1 && slot >= 8);
      if (none) *(v4u*)(ws + (int64_t)i * 16) = v4u{0, 0, 0, 0};
    }
    if (blockIdx.y == 0 && tid < 16 && gm_token<NM>(tid) >= T) exps[tid] = 0;
  }
}

// ---------------------------------------------------------------------------
// the products

struct GmArgs {
  const uint8_t* base;
  uint32_t head, range;
  int n_rows, K, T;
  const uint8_t* terms;
  float* y;
  int64_t ystride;
  const float* bias;
  const float* resid;  // may be y
  int npass, units;    // passes over K, units of a full pass
  int part_bytes;      // LDS bytes of a wave's part of a tile (GM_ROWS rows)
};

// The terms of one unit in registers.
template <int FMT, int NM>
struct Terms {
  b8 a[GM_PIECES<FMT>][NM];
};

__device__ __forceinline__ b8 gm_b8(v2u a, v2u b) { return __builtin_bit_cast(b8, v4u{a.x, a.y, b.x, b.y}); }

template <int N>
__device__ __forceinline__ v4f gm_mfma(const b8 (&x)[N], b8 w, v4f c) {
#pragma unroll
  for (int m = 0; m < N; ++m) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[m], w, c, 0, 0, 0);
  return c;
}

// y += unit (its bytes from o on in this lane's weight row) times the terms. MXFP4: times the tokens' scales as well (te, the
// A rows' scale exponents): a block scale alone may lie far outside the range of the product. The other formats' scales
// are f16, so the sums cannot leave fp32's range and the tokens' scales wait for the end. bf16 holds every code, a zero
// weight's as zero, but not Q4_K's with its sub-block's scale: those multiply the sums. (A block whose scale is infinite makes its row NaN: the terms' sums meet behind it.)
template <int FMT, int NM>
__device__ __forceinline__ void gm_unit(const LdsRow& R, const LdsRow& S0, int o, const Terms<FMT, NM>& X, int g, const int (&te)[4], v4f& y) {
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  auto add = [&](const v4f& d, float s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = fmaf(FMT == NSX_MXFP4 ? __builtin_amdgcn_ldexpf(d[i], -te[i]) : d[i], s, y[i]);
  };
  if constexpr (FMT == NSX_Q8_0) {
    const v2u w = R.words(o + 2);
    add(gm_mfma(X.a[0], gm_b8(sbytes4(w.x), sbytes4(w.y)), zero), nsx_h2f(R.get<uint16_t>(o)));
  } else if constexpr (FMT == NSX_Q4_0) {  // q - 8 as the upper half of a signed byte
    const uint32_t w = R.word(o + 2), lo = ((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u, hi = (w & 0xF0F0F0F0u) ^ 0x80808080u;
    add(gm_mfma(X.a[0], gm_b8(sbytes4(lo), sbytes4(hi)), zero), nsx_h2f(R.get<uint16_t>(o)));
  } else if constexpr (FMT == NSX_MXFP4) {
    const uint32_t w = R.word(o + 1);
    add(gm_mfma(X.a[0], gm_b8(fp4x4<0>(w), fp4x4<1>(w)), zero), nsx_mx_scale_half(R.get<uint8_t>(o)));
  } else if constexpr (FMT == NSX_Q4_K) {
    const v4u H = R.get<v4u>(o);  // d | dmin, scales[12]
    const uint32_t sc03 = H.y & 0x3F3F3F3Fu, sc47 = (H.w & 0x0F0F0F0Fu) | ((H.y >> 2) & 0x30303030u);
    const uint32_t mn03 = H.z & 0x3F3F3F3Fu, mn47 = ((H.w >> 4) & 0x0F0F0F0Fu) | ((H.z >> 2) & 0x30303030u);
    v4f acc = zero;
    auto sub = [&](const b8 (&x)[NM], uint32_t q0, uint32_t q1, float sc) {
      const v4f d = gm_mfma(x, gm_b8(nibbles4(q0), nibbles4(q1)), zero);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(sc, d[i], acc[i]);
    };
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) {  // sub-blocks 2 pr (low nibbles) and 2 pr + 1 (high ones)
      const uint32_t scw = pr < 2 ? sc03 : sc47;
      const v2u w = R.get<v2u>(o + 16 + 32 * pr + 8 * g);  // (rows of 16-byte pieces, 4-byte aligned: aligned here)
      sub(X.a[2 * pr], w.x & 0x0F0F0F0Fu, w.y & 0x0F0F0F0Fu, byte_of(scw, 2 * (pr & 1)));
      sub(X.a[2 * pr + 1], (w.x >> 4) & 0x0F0F0F0Fu, (w.y >> 4) & 0x0F0F0F0Fu, byte_of(scw, 2 * (pr & 1) + 1));
    }
    const v4f am = gm_mfma(X.a[8], gm_b8(bytes4(mn03), bytes4(mn47)), zero);
    add(acc, nsx_h2f(H.x & 0xFFFFu));
    add(am, -nsx_h2f(H.x >> 16));
  } else {  // Q6_K: a scale for every 16 elements; q - 32 as the upper six bits of a signed byte
    v4f acc = zero;
    uint32_t scw[4];  // the 16 scales
#pragma unroll
    for (int i = 0; i < 4; ++i) scw[i] = S0.word(o + 192 + 4 * i);
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) {
      const int h = hh >> 1, hl = hh & 1;
      const uint32_t qa = R.word(o + 64 * h + 16 * hl), qb = R.word(o + 64 * h + 32 + 16 * hl);
      const uint32_t qh = R.word(o + 128 + 32 * h + 16 * hl);
#pragma unroll
      for (int L = 0; L < 4; ++L) {
        const uint32_t ql = L & 1 ? qb : qa, low = L < 2 ? ql << 2 : ql >> 2;
        const uint32_t top = L == 0 ? qh << 6 : L == 1 ? qh << 4 : L == 2 ? qh << 2 : qh;
        const s4 b = __builtin_bit_cast(s4, sbytes4(((low & 0x3C3C3C3Cu) | (top & 0xC0C0C0C0u)) ^ 0x80808080u));
        v4f d = zero;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          const v4u x = __builtin_bit_cast(v4u, X.a[2 * hh + (L >> 1)][m]);
          const s4 xa = __builtin_bit_cast(s4, L & 1 ? v2u{x.z, x.w} : v2u{x.x, x.y});
          d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(xa, b, d, 0, 0, 0);
        }
        const float sc = sbyte_of(scw[(8 * h + hl + 2 * L) >> 2], (8 * h + hl + 2 * L) & 3);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(sc, d[i], acc[i]);
      }
    }
    add(acc, nsx_h2f(R.get<uint16_t>(o + 208)));
  }
}

__device__ __forceinline__ void gm_barrier() {  // LDS only: the next tile's loads stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int FMT, int NM, int MAXU>
__global__ __launch_bounds__(64 * gm_waves<FMT>(NM)) void gemv_mm_kernel(GmArgs a) {
  constexpr int UE = Unit<FMT>::E, UB = Unit<FMT>::B, W = gm_waves<FMT>(NM);
  constexpr int LOADS = (GM_ROWS * gm_pieces(MAXU * UB) + 63) / 64;  // 16-byte loads of a tile per lane
  extern __shared__ __align__(16) uint8_t gm_smem[];
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  uint8_t* buf = gm_smem + wave * a.part_bytes;
  constexpr int PART = GM_ROWS * GM_PS;
  float* parts = (float*)(gm_smem + W * a.part_bytes);  // [2][wave][A row][GM_PS]
  float* sums = parts + 2 * W * PART;                             // npass > 1: [tile of the group][16 token + row]
  const __amdgpu_buffer_rsrc_t rs = nsx_rsrc(a.base, a.range);
  const uint32_t rb = (uint32_t)(a.K / UE) * UB;
  const int ntiles = (a.n_rows + GM_ROWS - 1) / GM_ROWS;
  const int mine = (ntiles - 1 - (int)blockIdx.x) / (int)gridDim.x + 1;  // (the grid is at most ntiles)

  // This wave's part of a pass: units own0 .. own0 + own - 1, read as the MAXU units from u0 on (the neighbours' among
  // them have zero terms here), so that every place in LDS is a constant.
  constexpr int N16 = gm_pieces(MAXU * UB), PIECES = GM_ROWS * N16;
  int u0 = 0, own0 = 0, own = 0;
  LdsRow row, row0p;             // this lane's weight row in LDS, from its lane group's codes on; from its start
  uint32_t goff[LOADS];          // a tile's pieces: byte offset of piece lane + 64 q (in LDS at 16 (lane + 64 q))
  v4u stage[LOADS];
  Terms<FMT, NM> X[MAXU];
  int te[4];  // scale exponents of A rows 4 g .. 4 g + 3

  // Piece p of a tile: row p / N16 (at most rlast), bytes 16 (p % N16) .. from the dword that holds the first byte of
  // the wave's part of the row. The last pieces run into the next row. Lanes past the last piece repeat it.
  auto piece = [&](int q, int rlast) {
    const int p = min(lane + 64 * q, PIECES - 1), r = p / N16, c = p - r * N16;
    return ((a.head + (uint32_t)min(r, rlast) * rb + (uint32_t)u0 * UB) & ~3u) + (uint32_t)c * 16u;
  };
  auto slot = [&](int q) { return min(lane + 64 * q, PIECES - 1); };
  auto set_pass = [&](int pass) {
    const int all = a.K / UE, p0 = pass * a.units, pn = min(a.units, all - p0);
    const int per = pn / W, extra = pn % W;
    own = per + (wave < extra ? 1 : 0);
    own0 = p0 + wave * per + min(wave, extra);
    u0 = min(own0, all - MAXU);
    const uint32_t res = (a.head + (uint32_t)c16 * rb + (uint32_t)u0 * UB) & 3u;
    row.set(buf + c16 * N16 * 16, res, (FMT == NSX_Q8_0 ? 8u : 4u) * (uint32_t)g);
    row0p.set(buf + c16 * N16 * 16, res, 0);
#pragma unroll
    for (int q = 0; q < LOADS; ++q) goff[q] = piece(q, GM_ROWS - 1);
  };
  // A tile whose pieces could cross the end of the matrix (the last one): rows past it read its last row (their
  // results are not stored), and a piece that would cross it is moved back to end there, in LDS as well.
  const uint32_t rend = (a.range + 3u) & ~3u;
  auto row0 = [&](int i) { return ((int)blockIdx.x + i * (int)gridDim.x) * GM_ROWS; };
  auto at_end = [&](int i) { return (int64_t)(row0(i) + GM_ROWS) * rb + a.head + 64 > (int64_t)a.range; };
  auto rows_left = [&](int i) {  // (opaque: this rare case's places are not worth registers in the loop)
    int n = a.n_rows - 1 - row0(i);
    asm volatile("" : "+s"(n));
    return n;
  };
  // The loads of tile i (tiles start a multiple of 4 bytes apart: the pieces' places are the same in every tile).
  auto issue = [&](int i) {
    const uint32_t so = (uint32_t)row0(i) * rb;
    if (!at_end(i)) {
#pragma unroll
      for (int q = 0; q < LOADS; ++q)
        stage[q] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rs, goff[q], so, 0));
    } else {
      const int n = rows_left(i);
#pragma unroll
      for (int q = 0; q < LOADS; ++q)
        stage[q] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rs, min(piece(q, n) + so, rend - 16u), 0, 0));
    }
  };
  auto park = [&](int i) {  // the loaded pieces into LDS
    if (!at_end(i)) {
#pragma unroll
      for (int q = 0; q < LOADS; ++q) *(v4u*)(buf + 16 * slot(q)) = stage[q];
    } else {
      const int n = rows_left(i);
#pragma unroll
      for (int q = 0; q < LOADS; ++q) {
        const uint32_t at = piece(q, n) + (uint32_t)row0(i) * rb;
        __builtin_memcpy(buf + 16 * slot(q) - (at - min(at, rend - 16u)), &stage[q], 16);
      }
    }
  };
  // The terms of the pass (those of the neighbours' units zero).
  auto take_terms = [&]() {
    const v4u zero = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < MAXU; ++u) {
      const bool mine = (uint32_t)(u0 + u - own0) < (uint32_t)own;
#pragma unroll
      for (int pc = 0; pc < GM_PIECES<FMT>; ++pc)
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          const v4u t = *(const v4u*)(a.terms + ((((int64_t)(u0 + u) * GM_PIECES<FMT> + pc) * NM + m) * 64 + lane) * 16);
          X[u].a[pc][m] = __builtin_bit_cast(b8, mine ? t : zero);
        }
    }
  };
  const int32_t* exps = (const int32_t*)(a.terms + gm_terms_bytes<FMT>(a.K, NM));
#pragma unroll
  for (int i = 0; i < 4; ++i) te[i] = exps[4 * g + i];

  int flip = 0;
  for (int i0 = 0; i0 < mine; i0 += a.npass > 1 ? GM_GROUP : mine) {
    const int i1 = a.npass > 1 ? min(mine, i0 + GM_GROUP) : mine;
    for (int pass = 0; pass < a.npass; ++pass) {
      if (a.npass > 1 || i0 == 0) {
        set_pass(pass);
        issue(i0);
        take_terms();
      }
      // the sums of tile i (the waves' partials are in buffer `flip`)
      auto finish = [&](int i) {
        if ((int)threadIdx.x >= GM_ROWS * a.T) return;
        const int tok = threadIdx.x >> 4, r = threadIdx.x & 15, at = row0(i) + r;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
          const float* pw = parts + (flip * W + w) * PART + tok * GM_PS + r;
          v += NM == 1 ? (pw[0] + pw[5 * GM_PS]) + pw[10 * GM_PS] : NM == 2 ? pw[0] + pw[8 * GM_PS] : pw[0];
        }
        if (pass > 0) v += sums[(i - i0) * 256 + threadIdx.x];
        if (pass + 1 < a.npass) {
          sums[(i - i0) * 256 + threadIdx.x] = v;
        } else if (at < a.n_rows) {  // the reference's order: resid + (x @ W.T + bias)
          const int64_t o = (int64_t)tok * a.ystride + at;
          if (a.bias) v += a.bias[at];
          if (a.resid) v = a.resid[o] + v;
          a.y[o] = v;
        }
      };
      for (int i = i0; i < i1; ++i) {
        v4f y = {0.f, 0.f, 0.f, 0.f};
        park(i);
        if (i + 1 < i1) issue(i + 1);
        asm volatile("" ::: "memory");  // the wave's LDS operations run in order
        if (i > i0) {  // the tile before, behind this one's requests
          finish(i - 1);
          flip ^= 1;
        }
#pragma unroll
        for (int u = 0; u < MAXU; ++u) gm_unit<FMT, NM>(row, row0p, u * UB, X[u], g, te, y);
        // (the buffer that every wave has read by the barrier it met after the tile before)
        float* part = parts + (flip * W + wave) * PART;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(4 * g + r) * GM_PS + c16] = FMT == NSX_MXFP4 ? y[r] : __builtin_amdgcn_ldexpf(y[r], -te[r]);
        gm_barrier();
      }
      finish(i1 - 1);
      flip ^= 1;
    }
  }
}

template <int FMT, int NM, int E32>
int gm_launch(GmArgs a, hipStream_t st) {
  constexpr int MAXU = E32 * 32 / Unit<FMT>::E;
  a.part_bytes = GM_ROWS * gm_pieces(MAXU * Unit<FMT>::B) * 16;
  constexpr int W = gm_waves<FMT>(NM);
  const size_t lds = (size_t)W * a.part_bytes + 2 * W * GM_ROWS * GM_PS * sizeof(float) +
                     (a.npass > 1 ? GM_GROUP * 256 * sizeof(float) : 0);
  const void* k = (const void*)gemv_mm_kernel<FMT, NM, MAXU>;
  if (int rc = nsx_allow_lds(k, lds)) return rc;
  const int64_t grid = std::min<int64_t>(nsx_cdiv(a.n_rows, GM_ROWS), nsx_resident_workgroups(k, lds, 64 * W));
  hipLaunchKernelGGL((gemv_mm_kernel<FMT, NM, MAXU>), dim3((unsigned)grid), dim3(64 * W), lds, st, a);
  NSX_LAUNCHED();
  return NSX_OK;
}

// K in as few passes as the waves can hold, of equal length; the smallest kernel that holds one.
template <int FMT, int NM>
int gm_size(GmArgs a, hipStream_t st) {
  constexpr int UE = Unit<FMT>::E, CAP = gm_max_e32<FMT>(NM);
  const int all = a.K / UE;
  a.npass = (int)nsx_cdiv(all, gm_waves<FMT>(NM) * CAP * 32 / UE);
  a.units = (int)nsx_cdiv(all, a.npass);
  const int e32 = (int)nsx_cdiv(a.units, gm_waves<FMT>(NM)) * (UE / 32);
  if constexpr (UE == 32) {
    if (e32 <= 4) return gm_launch<FMT, NM, 4>(a, st);
    if (e32 <= 6) return gm_launch<FMT, NM, 6>(a, st);
  }
  if constexpr (CAP >= 8) {
    if (e32 <= 8) return gm_launch<FMT, NM, 8>(a, st);
  }
  if constexpr (UE == 32 && CAP >= 12) {
    if (e32 <= 12) return gm_launch<FMT, NM, 12>(a, st);
  }
  if constexpr (CAP >= 16) return gm_launch<FMT, NM, 16>(a, st);
  return nsx_fail(NSX_EINVAL, "K %d", a.K);
}

template <int FMT, int NM>
int gm_run(const void* raw, int64_t n_rows, int64_t K, const void* x, int x_dtype, int64_t T, float* y, const float* bias,
           const float* resid, uint8_t* ws, hipStream_t st) {
  // the terms, in as many parts as keep a thread's share small
  const unsigned parts = (unsigned)std::max<int64_t>(1, std::min<int64_t>(16, nsx_cdiv(K, 2048)));
  hipLaunchKernelGGL((gm_terms_kernel<FMT, NM>), dim3((unsigned)T, parts), dim3(256), 0, st, x, x_dtype, (int)K, (int)T, ws);
  NSX_LAUNCHED();
  const int64_t rb = K / Unit<FMT>::E * Unit<FMT>::B;
  const int64_t per = std::max<int64_t>(1, ((int64_t)1 << 31) / rb / GM_ROWS) * GM_ROWS;  // 32-bit byte offsets
  for (int64_t r0 = 0; r0 < n_rows; r0 += per) {
    const int64_t nr = std::min(per, n_rows - r0);
    const uint8_t* p = (const uint8_t*)raw + r0 * rb;
    const uintptr_t at = (uintptr_t)p & ~(uintptr_t)3;
    GmArgs a{};
    a.base = (const uint8_t*)at;
    a.head = (uint32_t)((uintptr_t)p - at);
    a.range = a.head + (uint32_t)(nr * rb);
    a.n_rows = (int)nr;
    a.K = (int)K;
    a.T = (int)T;
    a.terms = ws;
    a.y = y + r0;
    a.ystride = n_rows;
    a.bias = bias ? bias + r0 : nullptr;
    a.resid = resid ? resid + r0 : nullptr;
    if (int rc = gm_size<FMT, NM>(a, st)) return rc;
  }
  return NSX_OK;
}

int gm_mode(int64_t T) { return T <= 5 ? 1 : T <= 8 ? 2 : 3; }  // instructions per 32 elements

template <int FMT>
int gm_fmt(const void* raw, int64_t n_rows, int64_t K, const void* x, int x_dtype, int64_t T, float* y, const float* bias,
           const float* resid, uint8_t* ws, hipStream_t st) {
  switch (gm_mode(T)) {
    case 1: return gm_run<FMT, 1>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, ws, st);
    case 2: return gm_run<FMT, 2>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, ws, st);
    default: return gm_run<FMT, 3>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, ws, st);
  }
}

}  // namespace

int64_t nsx_gemv_mm_workspace(int t, int64_t n_rows, int64_t K, int64_t T) {
  if (T < 2 || T > GM_MAXT || K < 128) return 0;  // (a wave reads at least 4 blocks of 32)
  const int64_t least = T == 2 ? (t == NSX_Q6_K ? 64ll : t == NSX_Q4_K ? 24ll : 12ll)
                      : T <= 4 ? (t == NSX_Q6_K ? 24ll : 4ll) : 1ll;
  if (n_rows * K < least << 20) return 0;  // (nothing smaller is faster here)
  int64_t b = 0;
  switch (t) {
    case NSX_MXFP4: b = gm_terms_bytes<NSX_MXFP4>(K, gm_mode(T)); break;
    case NSX_Q4_0: b = gm_terms_bytes<NSX_Q4_0>(K, gm_mode(T)); break;
    case NSX_Q8_0: b = gm_terms_bytes<NSX_Q8_0>(K, gm_mode(T)); break;
    case NSX_Q4_K: b = gm_terms_bytes<NSX_Q4_K>(K, gm_mode(T)); break;
    case NSX_Q6_K: b = gm_terms_bytes<NSX_Q6_K>(K, gm_mode(T)); break;
    default: return 0;
  }
  return b + 64;
}

// Where this path is the faster one (us in a graph, VALU kernel / here). The VALU kernel's time grows with rows x K, with
// K x tokens where rows are few (a row's chain of units, once per 4 tokens) and in steps of its workgroups where K is
// small; this one's starts at its two launches and a tile's way through LDS, longer for the K-quants' wide blocks and for
// Q8_0 of 6 to 8 tokens (8 waves) outside K of 2048 .. 3072, where one pass of 12 units a wave holds all of it.
//  2 tokens: rows x K. Q4_0 2912 x 2880 9.4 / 10.1, 4119 x 2880 12.5 / 11.8; Q4_K 5825 x 2816 14.3 / 16.3, 8192 x 4096
//   22.1 / 18.2; Q6_K 8192 x 8192 38.7 / 35.1, 16384 x 4096 (two blocks a wave spill) 27.0 / 29.9, 32768 x 2048 29 / 23.
//  3, 4: Q4_0, MXFP4 from 4 Mi weights on (2048 x 2048 11.2 / 9.6); Q8_0 1024 x 4096 10.0 / 12.1, 2048 x 2048 10.7 / 9.6;
//   Q4_K 4096 x 1024 9.4 / 11.6, 2896 x 2048 13.2 / 13.1, 1448 x 4096 at 3 13.2 / 15.1, 512 x 8192 at 3 21 / 19.5.
//  5: Q4_0 1024 x 1024 7.6 / 8.5, 2048 x 512 7.3 / 8.1, 512 x 2048 11.0 / 9.4, 4096 x 256 8.9 / 8.0, 1448 x 1024 10 / 8.4;
//   Q4_K 1024 x 2048 10.0 / 12.6, 728 x 2816 12.0 / 13.5, 512 x 4096 16.1 / 14.7; Q6_K 728 x 2816 11.1 / 14.0.
//  6 to 8: MXFP4 1024 x 2048 10.1 / 10.7, 4096 x 256 11.7 / 8.1; Q8_0 1024 x 4096 at 6 18.3 / 20.6, at 8 24 / 20.9, 1024 x
//   2048 at 8 12.7 / 14.4, 1029 x 2880 21.9 / 12.4; Q4_K 2048 x 1024 at 6 12.6 / 13.0, 4096 x 512 10.9 / 11.7, 8192 x 256
//   15.8 / 12.3; Q6_K 1448 x 1024 7.7 / 9.9, 4096 x 256 11.6 / 8.9.
//  9 to 16: Q4_K 1024 x 1024 at 9 10.6 / 13.3, at 16 15 / 12; Q6_K the same, 9.7 / 10.9; the others gain from 1 Mi on.
static bool gm_pays(int t, int64_t n_rows, int64_t K, int64_t T) {
  const double n = (double)n_rows * K / (1 << 20);
  const int64_t kt = K * T;
  if (T == 2) return t != NSX_Q6_K || K <= 2048 || n >= 68;
  if (T <= 4) {
    if (t == NSX_Q8_0) return n >= 4.5 || kt >= 15000 || n_rows >= 2048;
    return t != NSX_Q4_K || n >= 6 || kt >= 24000 || n_rows >= 10000;
  }
  if (T > 8) return n >= 1.25 || (t != NSX_Q4_K && t != NSX_Q6_K) || T >= 12 || kt >= 15000 || n_rows >= 2048;
  switch (t) {
    case NSX_Q4_K: return n >= 2.25 || kt >= (T == 5 ? 20000 : 26000) || n_rows >= 5500;
    case NSX_Q6_K: return n >= 2.25 || kt >= 20000 || n_rows >= 2800;
    case NSX_Q8_0:
      if (T > 5) return n >= 4.25 || kt >= (K > 2048 && K <= 3072 ? 17000 : 26000) || n_rows >= 2048;
      break;
    case NSX_MXFP4:
      if (T > 5) return n >= 2.25 || kt >= 15000 || n_rows >= 2800;
      break;
  }
  return n >= 1.25 || kt >= (T == 5 ? 10000 : 15000) || n_rows >= 2800;
}

int nsx_gemv_mm_takes(int t, int64_t n_rows, int64_t K, int64_t T) {
  return nsx_gemv_mm_workspace(t, n_rows, K, T) > 0 && gm_pays(t, n_rows, K, T);
}

int nsx_gemv_mm(int t, const void* raw, int64_t n_rows, int64_t K, const void* x, int x_dtype, int64_t T, float* y,
                const float* bias, const float* resid, void* ws, hipStream_t st) {
  uint8_t* w = (uint8_t*)ws;
  switch (t) {
    case NSX_MXFP4: return gm_fmt<NSX_MXFP4>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, w, st);
    case NSX_Q4_0: return gm_fmt<NSX_Q4_0>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, w, st);
    case NSX_Q8_0: return gm_fmt<NSX_Q8_0>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, w, st);
    case NSX_Q4_K: return gm_fmt<NSX_Q4_K>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, w, st);
    case NSX_Q6_K: return gm_fmt<NSX_Q6_K>(raw, n_rows, K, x, x_dtype, T, y, bias, resid, w, st);
  }
  return nsx_fail(NSX_ENOTIMPL, "ggml type %d", t);
}
