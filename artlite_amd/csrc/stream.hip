// The streamed small tiles: the experts' products for tiles of at most 64 rows, on the fp16 or bf16 MFMA (16x16x32) over
// the blocks' integer codes.
//
// Numerics. A block's codes are exact in fp16 (1024 + code) and in bf16 (128 + code, codes.h); the activations are the
// prefill's scaled fp16 rows, or bf16 planes (bf16 x exactly; fp32 x and h as hi + lo, 2^-17). Per 32-value group one
// MFMA of the activations against a constant -offset gives the C input that takes the codes' offset off, then one per
// plane against the codes, so p = sum code x in fp32; the group's fp32 scale (and min) is applied to the sum:
// acc += d p. (No weight is rounded, where the prefill tiles round d (q - 8) to fp16. A row of A with a non-finite value
// gives NaN, as on the decode GEMV.)
//
// What bounds it: HBM, then the VALU: at 8 rows an expert (128 experts, Q4_0) gate / up reads its 226 MB in 57 us,
// 4.0 TB/s (110 us on the prefill tiles), the down its 113 MB in 34 (63). A wave's 16 weight rows of a group take about 14
// to 30 VALU instructions (the codes to fp16, the scale, 4 FMAs) whatever the tile's rows up to 16, where the decode GEMV
// takes about 22 per row of A and the prefill tiles a step's fixed cost per 64 values of K. The codes are read as aligned
// dwords: 18-byte blocks read in unaligned pieces took gate / up from 57 to 79 us.
//
// A tile of 64 rows takes a weight's codes to fp16 and its scale once for up to 64 rows of A, where two tiles of 32 do both
// again: at 40 rows an expert the Q4_0 layer takes 213 us in tiles of 64, 242 in tiles of 32 and 229 on the prefill tiles
// (Q4_K: 232, 254, 291; Q8_0: 251, 298, 289). It costs LDS: 4-bit formats then have 1 workgroup of 8 waves a CU.
//
// Shape of the work. An item is a tile (16, 32 or 64 rows of A at most, one expert's; its products run over as many
// 16-row column blocks as it fills) times 16 WAVES rows of gate and the
// same of up (plain products: 32 WAVES rows); persistent workgroups take items in turn, tile-major. A wave has 2 blocks of
// 16 weight rows (SwiGLU: gate and up of the same rows, so that h forms in its registers) and streams them, a step of SV
// values of K at a time, into a ring of LDS slots of its own; the tile's activations for the step, which all waves
// read, come into a ring the workgroup shares. Every load is a DMA (global_load_lds, by asm, so that the compiler does
// not wait for it), a step ahead, across items. One barrier a step: past it the step's activations (every wave's part)
// have landed and the slot of the step before is free.
// Activation rows sit in LDS as 16-byte chunks XOR-swizzled by row (the 16 rows a lane group reads in different banks).
// MFMA layout (16x16x32): lane l holds A row l % 16 (a row of the tile) and B column l % 16 (a weight row), both with K
// values 8 (l / 16) .. + 8; C column l % 16, rows 4 (l / 16) .. + 4: a lane's four sums share its weight row's scale.
#include "stream.h"

#include "codes.h"
#include "experts.h"

#include <algorithm>
#include <utility>

namespace artlite {

namespace {

template <typename F, int... I>
__device__ __forceinline__ void st_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void st_for(F&& f) {
  st_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int N>
__device__ __forceinline__ void st_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
// every LDS read of the wave done, then the workgroup barrier
__device__ __forceinline__ void st_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ uint32_t st_lds_addr(const void* p) {
  return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}

// every LDS read of the wave done (the slot they read may be loaded again)
__device__ __forceinline__ void st_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// One DMA of 16 bytes per lane from the lane's address into LDS at lds (uniform) + 16 lane (M0 carries the LDS address;
// no compiler-generated code of this kernel uses it)
__device__ __forceinline__ void st_dma(const uint8_t* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory");
}
// the same from a uniform base and the lane's 32-bit byte offset
__device__ __forceinline__ void st_dma(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
               : "memory");
}

// Ring slots: two, a step's loads in flight while the one before computes (a third measured the same or slower: Q4_0
// gate / up at 8 rows an expert 57.5 against 53.9 us)
constexpr int SLOTS = 2;

// Per format: the values of K of a step, a row's bytes of it and their LDS stride (whole 16-byte chunks: Q8_0's 136
// bytes are loaded with the 8 after them, so that two workgroups a CU fit)
template <int QT>
struct SF {
  static constexpr int SV = QT == ARTLITE_Q8_0 ? 128 : 256;
  static constexpr int NG = SV / 32;
  static constexpr int BYTES = SV / (32 * Fmt<QT>::GPB) * Fmt<QT>::BLOCK_BYTES;
  static constexpr int CH = (BYTES + 15) / 16, STRIDE = 16 * CH;
};

// A launch's shape: WAVES, tiles of 16 NC rows of A
template <int QT, bool SWIGLU, int WAVES, int NC>
struct SL {
  using F = SF<QT>;
  static constexpr int NBK = 2;                                   // 16-row blocks of a wave
  static constexpr int RBW = SWIGLU ? 16 * WAVES : 32 * WAVES;    // rows of N per item
  static constexpr int THREADS = 64 * WAVES;
  static constexpr int WCH = NBK * 16 * F::CH, NI = (WCH + 63) / 64, LAST = WCH - 64 * (NI - 1);
  static constexpr int WSLOT = WCH * 16;                          // bytes of a wave's slot
  static constexpr int RCH = F::SV / 8;                           // chunks of an activation row's step
  static constexpr int ACOL = 16 * RCH * 16, ASLOT = NC * ACOL;  // (a column block's activations, a slot's)
  static constexpr int NA = ACOL / 1024 / WAVES;                  // activation DMAs of a wave a column block's step
  static constexpr int LDS = SLOTS * (WAVES * WSLOT + ASLOT);     // (then the item table)
  static constexpr int ENTRY = 4 + 16 * NC;                       // ints of an item's entry (below)
};

// what a step takes of a weight row beyond its codes: the super-block's header, read once a step
template <int QT>
struct Hdr {
  u32x4 h;
  uint32_t d;
  __device__ __forceinline__ void read(const uint8_t* row) {
    if constexpr (QT == ARTLITE_Q4_K || QT == ARTLITE_Q5_K) {
      h = *reinterpret_cast<const u32x4*>(row);
    } else if constexpr (QT == ARTLITE_Q6_K) {
      h = *reinterpret_cast<const u32x4*>(row + 192);
      d = lds_u16(row + 208);
    }
  }
};

// eight code bytes -> four dwords of fp16 1024 + c
__device__ __forceinline__ u32x4 half8(uint32_t v0, uint32_t v1) {
  return u32x4{__builtin_amdgcn_perm(0x64646464u, v0, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, v0, 0x04030402u),
               __builtin_amdgcn_perm(0x64646464u, v1, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, v1, 0x04030402u)};
}

// the formats whose code bytes take all 8 bits (Q8_0's q + 128, the IQ4 values + 128)
template <int QT>
constexpr bool byte_codes = QT == ARTLITE_Q8_0 || QT == ARTLITE_IQ4_NL || QT == ARTLITE_IQ4_XS;

// B operand of group g of a row's step for lane group lg (values 8 lg .. + 8): the 8 codes in A's type and the scales
// (as codes.h's b_operand)
template <int QT, bool H>
__device__ __forceinline__ u32x4 st_operand(const uint8_t* row, const Hdr<QT>& hd, int g, int lg, float& sc, float& mn,
                                            float& sc2) {
  uint32_t u0, u1;
  if constexpr (QT == ARTLITE_Q4_K || QT == ARTLITE_Q5_K) {
    const int sh8 = 8 * (g & 3);
    uint32_t q6, m6;
    if (g < 4) {
      q6 = (hd.h[1] >> sh8) & 63;
      m6 = (hd.h[2] >> sh8) & 63;
    } else {
      q6 = ((hd.h[3] >> sh8) & 15) | (((hd.h[1] >> (sh8 + 6)) & 3) << 4);
      m6 = ((hd.h[3] >> (sh8 + 4)) & 15) | (((hd.h[2] >> (sh8 + 6)) & 3) << 4);
    }
    sc = __fmul_rn(h2f(hd.h[0] & 0xFFFFu), float(q6));
    mn = __fmul_rn(h2f(hd.h[0] >> 16), float(m6));
    const uint8_t* qs = row + (QT == ARTLITE_Q5_K ? 48 : 16) + 32 * (g >> 1) + 8 * lg;
    const int sh = 4 * (g & 1);
    const uint2 q = *reinterpret_cast<const uint2*>(qs);
    u0 = (q.x >> sh) & 0x0F0F0F0Fu, u1 = (q.y >> sh) & 0x0F0F0F0Fu;
    if constexpr (QT == ARTLITE_Q5_K) {
      const uint2 b = *reinterpret_cast<const uint2*>(row + 16 + 8 * lg);
      u0 |= ((b.x >> g) & 0x01010101u) << 4;
      u1 |= ((b.y >> g) & 0x01010101u) << 4;
    }
  } else if constexpr (QT == ARTLITE_Q6_K) {
    const int h = g >> 2, jj = g & 3;
    const float d = h2f(hd.d);
    const uint32_t s2 = hd.h[g >> 1] >> (16 * (g & 1));
    sc = __fmul_rn(float(int8_t(s2 & 0xFFu)), d);
    sc2 = __fmul_rn(float(int8_t((s2 >> 8) & 0xFFu)), d);
    const uint2 ql = *reinterpret_cast<const uint2*>(row + 64 * h + 32 * (jj & 1) + 8 * lg);
    const uint2 qh = *reinterpret_cast<const uint2*>(row + 128 + 32 * h + 8 * lg);
    const int sh = jj < 2 ? 0 : 4;
    u0 = ((ql.x >> sh) & 0x0F0F0F0Fu) | (((qh.x >> (2 * jj)) & 0x03030303u) << 4);
    u1 = ((ql.y >> sh) & 0x0F0F0F0Fu) | (((qh.y >> (2 * jj)) & 0x03030303u) << 4);
  } else if constexpr (QT == ARTLITE_Q8_0) {
    // (34-byte blocks, a pair of groups 17 dwords: the first's codes start 2 bytes into dword 0, the second's at dword
    // 9, its scale the high half of dword 8)
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row + 68 * (g >> 1));
    const uint32_t* q = p + 2 * lg;
    if (g & 1) {
      sc = h2f(p[8] >> 16);
      u0 = q[9], u1 = q[10];
    } else {
      const uint32_t w0 = q[0], w1 = q[1], w2 = q[2];
      sc = h2f(p[0] & 0xFFFFu);
      u0 = __builtin_amdgcn_alignbit(w1, w0, 16), u1 = __builtin_amdgcn_alignbit(w2, w1, 16);
    }
    u0 ^= 0x80808080u, u1 ^= 0x80808080u;
  } else if constexpr (QT == ARTLITE_Q3_K) {
    const int n = g >> 2, j = g & 3;
    const float d = h2f(lds_u16(row + 108));
    sc = __fmul_rn(d, float(q3k_scale(row + 96, 2 * g)));
    sc2 = __fmul_rn(d, float(q3k_scale(row + 96, 2 * g + 1)));
    const uint2 q = *reinterpret_cast<const uint2*>(row + 32 + 32 * n + 8 * lg);
    const uint2 m = *reinterpret_cast<const uint2*>(row + 8 * lg);
    u0 = ((q.x >> (2 * j)) & 0x03030303u) | (((m.x >> (4 * n + j)) & 0x01010101u) << 2);
    u1 = ((q.y >> (2 * j)) & 0x03030303u) | (((m.y >> (4 * n + j)) & 0x01010101u) << 2);
  } else if constexpr (QT == ARTLITE_Q4_0 || QT == ARTLITE_IQ4_NL) {
    // (18-byte blocks in aligned dwords, a pair of groups 9 of them: the first's codes start 2 bytes into dword 0, the
    // second's at dword 5, its scale the high half of dword 4)
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row + 36 * (g >> 1));
    const uint32_t* q = p + 2 * (lg & 1);
    const int sh = 4 * (lg >> 1);
    if (g & 1) {
      sc = h2f(p[4] >> 16);
      u0 = q[5], u1 = q[6];
    } else {
      const uint32_t w0 = q[0], w1 = q[1], w2 = q[2];
      sc = h2f(p[0] & 0xFFFFu);
      u0 = __builtin_amdgcn_alignbit(w1, w0, 16), u1 = __builtin_amdgcn_alignbit(w2, w1, 16);
    }
    u0 = (u0 >> sh) & 0x0F0F0F0Fu, u1 = (u1 >> sh) & 0x0F0F0F0Fu;
    if constexpr (byte_codes<QT>) u0 = iq4_bytes(u0), u1 = iq4_bytes(u1);
  } else {  // Q4_1's 20-byte blocks (d, then m: w = d q + m, mn = -m); IQ4_XS: a group's 16 bytes of the padded block
    const uint8_t* qs;
    if constexpr (QT == ARTLITE_IQ4_XS) {
      const int ls = ((row[4 + g / 2] >> (4 * (g & 1))) & 15) | (((int(lds_u16(row + 2)) >> (2 * g)) & 3) << 4);
      sc = __fmul_rn(h2f(lds_u16(row)), float(ls - 32));
      qs = row + 16 + 16 * g;
    } else {
      sc = h2f(lds_u16(row + 20 * g));
      mn = -h2f(lds_u16(row + 20 * g + 2));
      qs = row + 20 * g + 4;
    }
    const int sh = 4 * (lg >> 1);
    u0 = (lds_u32(qs + 8 * (lg & 1)) >> sh) & 0x0F0F0F0Fu;
    u1 = (lds_u32(qs + 4 + 8 * (lg & 1)) >> sh) & 0x0F0F0F0Fu;
    if constexpr (byte_codes<QT>) u0 = iq4_bytes(u0), u1 = iq4_bytes(u1);
  }
  return H ? half8(u0, u1) : byte_codes<QT> ? byte8(u0, u1) : nib8(u0, u1);
}

// the offset of the codes' encoding: in bf16 (Fmt::OFF) 128 + code, or the code itself where it takes all 8 bits; in
// fp16 1024 + code
template <int QT, bool H>
constexpr float code_off() {
  return Fmt<QT>::OFF + (!H ? 0.0f : byte_codes<QT> ? 1024.0f : 896.0f);
}
// the offset's negative, twice, in A's type (exact)
template <int QT, bool H>
constexpr uint32_t off_pair() {
  const uint32_t u = H ? uint32_t(__builtin_bit_cast(uint16_t, _Float16(-code_off<QT, H>())))
                       : __builtin_bit_cast(uint32_t, -code_off<QT, H>()) >> 16;
  return u | (u << 16);
}

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
template <bool H>
__device__ __forceinline__ f32x4 st_mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (H)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  else
    return mfma(a, b, c);
}

// Group g of a step: the wave's two blocks' sums over it, for NC column blocks of 16 rows of A. row: the lane's weight
// rows in LDS (one per block); x: the lane's activations of the group, by column block and plane.
template <int QT, bool H, int AP, int NC>
__device__ __forceinline__ void st_group(const uint8_t* const (&row)[2], const Hdr<QT> (&hd)[2], const u32x4 (&x)[NC][AP],
                                         int g, int lg, f32x4 (&acc)[NC][2]) {
  using F = Fmt<QT>;
  constexpr uint32_t OFFC = off_pair<QT, H>();
  const u32x4 zero{0, 0, 0, 0}, off{OFFC, OFFC, OFFC, OFFC};
  const f32x4 z{0, 0, 0, 0};
  // (16-value scales: lane groups 0, 1 hold the group's first 16 values, 2, 3 its second 16: a product per half, the other
  // half's activations 0)
  constexpr int HV = F::SUB16 ? 2 : 1;
  u32x4 xh[NC][HV][AP];
  f32x4 cin[NC][HV];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int h = 0; h < HV; h++) {
      cin[c][h] = z;
#pragma unroll
      for (int pl = AP - 1; pl >= 0; pl--) {
        xh[c][h][pl] = HV == 1 || (lg < 2) == (h == 0) ? x[c][pl] : zero;
        cin[c][h] = st_mfma<H>(xh[c][h][pl], off, cin[c][h]);
      }
    }
#pragma unroll
  for (int b = 0; b < 2; b++) {
    float sc, mn = 0.0f, sc2 = 0.0f;
    const u32x4 q = st_operand<QT, H>(row[b], hd[b], g, lg, sc, mn, sc2);
    const float m1 = mn * (1.0f / code_off<QT, H>());
#pragma unroll
    for (int c = 0; c < NC; c++) {
      f32x4 p[HV];
#pragma unroll
      for (int h = 0; h < HV; h++) {
        p[h] = cin[c][h];
#pragma unroll
        for (int pl = AP - 1; pl >= 0; pl--) p[h] = st_mfma<H>(xh[c][h][pl], q, p[h]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        acc[c][b][i] = __builtin_fmaf(sc, p[0][i], acc[c][b][i]);
        if (HV == 2) acc[c][b][i] = __builtin_fmaf(sc2, p[HV - 1][i], acc[c][b][i]);
        if (F::MIN) acc[c][b][i] = __builtin_fmaf(m1, cin[c][0][i], acc[c][b][i]);
      }
    }
  }
}

template <int QT, bool SWIGLU, int WAVES, int NC>
__global__ __launch_bounds__(64 * WAVES) __attribute__((
    amdgpu_waves_per_eu(2, QT == ARTLITE_Q8_0 ? 8 : 2))) void k_stream(const StreamArgs a) {
  using F = SF<QT>;
  using L = SL<QT, SWIGLU, WAVES, NC>;
  constexpr int BM = 16 * NC;
  static_assert(L::NA * 1024 * WAVES == L::ACOL, "whole activation DMAs");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lg = lane >> 4,
            lr = lane & 15;
  // the workgroup's items blockIdx.x, + G, ..., in a table: the expert, first sorted row, rows, first row of N, then the
  // A rows of its BM rows (the last valid one repeated)
  int* table = reinterpret_cast<int*>(lds + L::LDS);
  const int G = gridDim.x;
  const int n_tiles = *a.n_tiles, NB = (a.N + L::RBW - 1) / L::RBW;
  const int total = n_tiles * NB, n_my = int(blockIdx.x) < total ? (total - 1 - int(blockIdx.x)) / G + 1 : 0;
  if (n_my == 0) return;
  for (int j = tid / BM; j < n_my; j += L::THREADS / BM) {
    const int t = tid % BM, it = int(blockIdx.x) + j * G, tile = it / NB;
    // (an expert's next tile, or the next expert's first, starts where this one ends)
    const int e = a.tiles[2 * tile], s0 = a.tiles[2 * tile + 1], end = tile + 1 < n_tiles ? a.tiles[2 * tile + 3] : a.rows;
    const int m = min(BM, end - s0), s = s0 + min(t, m - 1);
    int* o = table + j * L::ENTRY;
    o[4 + t] = a.row_a ? a.row_a[s] : s;
    if (t == 0) {
      o[0] = e;
      o[1] = s0;
      o[2] = m;
      o[3] = (it - tile * NB) * L::RBW;
    }
  }
  __syncthreads();

  uint8_t* const wl = lds + wv * (SLOTS * L::WSLOT);              // the wave's weight slots
  uint8_t* const al = lds + WAVES * SLOTS * L::WSLOT;             // the workgroup's activation slots
  const uint32_t wl0 = __builtin_amdgcn_readfirstlane(st_lds_addr(wl)), al0 = __builtin_amdgcn_readfirstlane(st_lds_addr(al));

  // ---- the issue side: the step next to be loaded (item iq, step iu of it)
  int iq = 0, iu = 0, islot = 0, icol = 0;
  const int steps = (a.K + F::SV - 1) / F::SV, kch = a.K / 8;
  const uint8_t* wp[L::NI];  // the lane's weight sources of the step
  uint32_t ao[NC][L::NA];    // the lane's activation sources: its row's byte offset
  auto open_item = [&]() {
    const int* o = table + iq * L::ENTRY;
    const int e = __builtin_amdgcn_readfirstlane(o[0]), n0 = __builtin_amdgcn_readfirstlane(o[3]);
    icol = (__builtin_amdgcn_readfirstlane(o[2]) + 15) / 16;
    const int64_t eo = int64_t(e) * a.expert_bytes;
#pragma unroll
    for (int i = 0; i < L::NI; i++) {
      const int q = min(64 * i + lane, L::WCH - 1), r = q / F::CH, c = q - r * F::CH;
      const int n = min(n0 + (SWIGLU ? 16 * wv + (r & 15) : 32 * wv + r), a.N - 1);  // (rows past N: the last again)
      wp[i] = (SWIGLU && r >= 16 ? a.w[1] : a.w[0]) + eo + int64_t(n) * a.row_bytes + 16 * c;
    }
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
#pragma unroll
      for (int i = 0; i < L::NA; i++) {
        const int c = 64 * (wv + WAVES * i) + lane;  // (the LDS chunk within the column block: row, chunk of the row)
        ao[cb][i] = uint32_t(o[4 + 16 * cb + c / L::RCH]) * uint32_t(a.K) * 2;
      }
  };
  auto issue = [&]() {
    if (iq >= n_my) return;
    const uint32_t wd = __builtin_amdgcn_readfirstlane(wl0 + islot * L::WSLOT),
                   ad = __builtin_amdgcn_readfirstlane(al0 + islot * L::ASLOT);
#pragma unroll
    for (int i = 0; i < L::NI; i++) {
      if (i < L::NI - 1 || L::LAST == 64 || lane < L::LAST) st_dma(wp[i], wd + 1024 * i);
      wp[i] += F::BYTES;
    }
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
      if (cb < icol)
#pragma unroll
        for (int i = 0; i < L::NA; i++) {
          const int q = wv + WAVES * i, c = 64 * q + lane, row = c / L::RCH;
          const int k = min(iu * L::RCH + ((c % L::RCH) ^ row), kch - 1);  // (chunks past K: its last one, unread)
          st_dma(a.a, ao[cb][i] + 16 * k, ad + cb * L::ACOL + 1024 * q);
        }
    islot ^= 1;
    if (++iu == steps) {
      iu = 0;
      if (++iq < n_my) open_item();
    }
  };
  open_item();
  issue();

  // ---- the products
  // (the lane's chunk of group 0 in a column block; group g's: ^ 64 g)
  const uint32_t xo = lr * L::RCH * 16 + (((lg ^ (lr & 3)) | (lr & 12)) * 16);
  int slot = 0;
  // an item of C column blocks
  auto run = [&](auto cc, int s0, int m, int n0) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    f32x4 acc[C][2];
    float2 fr[C][4];  // (the factors of the lane's output rows)
#pragma unroll
    for (int c = 0; c < C; c++) {
      acc[c][0] = acc[c][1] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 4; i++) fr[c][i] = a.row_scale[s0 + min(16 * c + 4 * lg + i, m - 1)];
    }
    for (int u = 0; u < steps; u++) {
      st_wait<0>();  // (this step's loads, the only ones in flight)
      st_barrier();
      issue();
      const uint8_t* ws = wl + slot * L::WSLOT;
      const uint8_t* xs = al + slot * L::ASLOT;
      const uint8_t* row[2] = {ws + lr * F::STRIDE, ws + (16 + lr) * F::STRIDE};
      Hdr<QT> hd[2];
      hd[0].read(row[0]);
      hd[1].read(row[1]);
      const int ng = min(F::NG, a.K / 32 - u * F::NG);
      auto group = [&](int g) __attribute__((always_inline)) {
        u32x4 x[C][1];
#pragma unroll
        for (int c = 0; c < C; c++) x[c][0] = *reinterpret_cast<const u32x4*>(xs + c * L::ACOL + (xo ^ (64 * g)));
        st_group<QT, true, 1, C>(row, hd, x, g, lg, acc);
      };
      if (ng == F::NG)
        st_for<F::NG>([&](auto gc) __attribute__((always_inline)) { group(decltype(gc)::value); });
      else
        for (int g = 0; g < ng; g++) group(g);
      slot ^= 1;
    }
    // the outputs: lane output i is tile row 16 c + 4 lg + i, column n0 + 16 wv + lr (plain: block b's, n0 + 32 wv + 16 b
    // + lr)
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int t = 16 * c + 4 * lg + i;
        if (t >= m) continue;
        const float2 f = fr[c][i];
        if constexpr (SWIGLU) {
          const int n = n0 + 16 * wv + lr;
          if (n < a.N) {
            const float gv = acc[c][0][i] * f.x, h = gv / (1.0f + __expf(-gv)) * (acc[c][1][i] * f.x);
            a.h[int64_t(s0 + t) * a.N + n] = __builtin_bit_cast(uint16_t, _Float16(h * f.y));
          }
        } else {
#pragma unroll
          for (int b = 0; b < 2; b++) {
            const int n = n0 + 32 * wv + 16 * b + lr;
            if (n < a.N) a.y16[int64_t(s0 + t) * a.N + n] = __builtin_bit_cast(uint16_t, _Float16(acc[c][b][i] * f.y));
          }
        }
      }
  };
  for (int j = 0; j < n_my; j++) {
    const int* o = table + j * L::ENTRY;
    const int s0 = __builtin_amdgcn_readfirstlane(o[1]), m = __builtin_amdgcn_readfirstlane(o[2]),
              n0 = __builtin_amdgcn_readfirstlane(o[3]);
    if (NC == 1 || m <= 16)
      run(std::integral_constant<int, 1>{}, s0, m, n0);
    else if (NC == 2 || m <= 32)
      run(std::integral_constant<int, (NC < 2 ? NC : 2)>{}, s0, m, n0);
    else if (m <= 48)
      run(std::integral_constant<int, (NC < 3 ? NC : 3)>{}, s0, m, n0);
    else
      run(std::integral_constant<int, NC>{}, s0, m, n0);
  }
}

// The dense rows of a shared expert beside decode-sized or streamed routed ones (a few to 256 tokens; any number where it has
// no prefill tiles), on bf16 planes: at a few tokens a product whose items are too few for the device, so a workgroup takes 16 weight rows of gate and of up (plain: 32 rows) of a tile and
// its 8 waves split K: wave w streams steps w, w + 8, ... of every row by DMA into its LDS slot, its activations come
// from memory (L2) to registers, and the waves' sums meet in LDS, added in wave order by wave 0, which writes the
// outputs. What bounds it is latency: a launch, two memory round trips, a step or two of products and the exchange
// (8 tokens, 2816 wide, Q4_K: a workgroup of four waves over all of K 15 and 23 us, split 7 and 9).
template <int QT, bool SWIGLU, int AP>
__global__ __launch_bounds__(512) void k_stream_few(const StreamFewArgs a) {
  using F = SF<QT>;
  using L = SL<QT, SWIGLU, 1, 1>;  // (a wave's slot and its DMAs)
  constexpr int W = 8;
  __shared__ __attribute__((aligned(16))) uint8_t slots[W * L::WSLOT];
  __shared__ f32x4 red[W - 1][2][WAVE];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lg = lane >> 4,
            lr = lane & 15;
  const int n0 = int(blockIdx.x) * L::RBW, s0 = int(blockIdx.y) * 16, m = min(16, a.rows - s0);
  const int steps = (a.K + F::SV - 1) / F::SV;
  uint8_t* const ws = slots + wv * L::WSLOT;
  const uint32_t wd = __builtin_amdgcn_readfirstlane(st_lds_addr(ws));
  const uint8_t* wp[L::NI];
#pragma unroll
  for (int i = 0; i < L::NI; i++) {
    const int q = min(64 * i + lane, L::WCH - 1), r = q / F::CH, c = q - r * F::CH;
    const int n = min(n0 + (SWIGLU ? (r & 15) : r), a.N - 1);  // (rows past N: the last again)
    wp[i] = (SWIGLU && r >= 16 ? a.w[1] : a.w[0]) + int64_t(n) * a.row_bytes + 16 * c;
  }
  const int64_t xo = int64_t(s0 + min(lr, m - 1)) * a.K + 8 * lg;
  f32x4 sum[1][2] = {{f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}}};
  f32x4(&acc)[2] = sum[0];
  for (int u = wv; u < steps; u += W) {
    st_reads_done();  // (of the slot, by the step before)
#pragma unroll
    for (int i = 0; i < L::NI; i++)
      if (i < L::NI - 1 || L::LAST == 64 || lane < L::LAST) st_dma(wp[i] + int64_t(u) * F::BYTES, wd + 1024 * i);
    u32x4 x[F::NG][1][AP];
#pragma unroll
    for (int g = 0; g < F::NG; g++) {
      const int64_t k = xo + min(u * F::SV + 32 * g, a.K - 32);  // (groups past K: its last, unused)
      x[g][0][0] = *reinterpret_cast<const u32x4*>(a.a + k);
      if constexpr (AP == 2) x[g][0][AP - 1] = *reinterpret_cast<const u32x4*>(a.a_lo + k);
    }
    st_wait<0>();
    const uint8_t* row[2] = {ws + lr * F::STRIDE, ws + (16 + lr) * F::STRIDE};
    Hdr<QT> hd[2];
    hd[0].read(row[0]);
    hd[1].read(row[1]);
    const int ng = min(F::NG, a.K / 32 - u * F::NG);
    st_for<F::NG>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
      if (g < ng) st_group<QT, false, AP, 1>(row, hd, x[g], g, lg, sum);
    });
  }
  if (wv)
#pragma unroll
    for (int b = 0; b < 2; b++) red[wv - 1][b][lane] = acc[b];
  __syncthreads();
  if (wv) return;
#pragma unroll
  for (int w = 0; w < W - 1; w++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[b] += red[w][b][lane];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int t = 4 * lg + i;
    if (t >= m) continue;
    if constexpr (SWIGLU) {
      const int n = n0 + lr;
      if (n < a.N) {
        const float gv = acc[0][i], h = gv / (1.0f + expf(-gv)) * acc[1][i];
        const uint32_t hi = f32_to_bf16(h);
        const int64_t at = int64_t(s0 + t) * a.N + n;
        a.h_hi[at] = uint16_t(hi);
        a.h_lo[at] = uint16_t(f32_to_bf16(h - bf16_to_f32(hi)));
      }
    } else {
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int n = n0 + 16 * b + lr;
        if (n < a.N) a.y[int64_t(s0 + t) * a.N + n] = acc[b][i];
      }
    }
  }
}

// A launch's persistent workgroups and the entries of their item tables, for `items` items: as many workgroups a CU (two
// at most, or three of Q8_0's, whose steps are half as long) as LDS holds with tables that take every item; false: none.
// (At 8 rows an expert Q4_0's gate / up took 54 us with two workgroups of three items a CU and 67 us with three of two;
// Q8_0's, 2880 wide, 106 us with two and 97 with three.)
template <int QT, bool SWIGLU, int WAVES, int NC>
bool stream_grid(int64_t items, int cus, int64_t& grid, int64_t& entries) {
  using L = SL<QT, SWIGLU, WAVES, NC>;
  constexpr int GRAIN = 1280;  // (the unit of LDS allocation)
  for (int c = QT == ARTLITE_Q8_0 ? 3 : 2; c >= 1; c--) {
    const int room = LDS_BYTES / c / GRAIN * GRAIN - L::LDS, q = room > 0 ? room / (L::ENTRY * 4) : 0;
    grid = std::min<int64_t>(items, int64_t(c) * cus);
    entries = (items + grid - 1) / grid;
    if (entries <= q) return true;
  }
  return false;
}

// (0: set-up failed)
int device_cus() {
  static const int cus = [] {
    int dev = 0, n = 0;
    return hipGetDevice(&dev) == hipSuccess &&
                   hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess
               ? n
               : 0;
  }();
  return cus;
}

template <int QT, bool SWIGLU, int WAVES, int NC>
int launch_t(const StreamArgs& a, bool dry, hipStream_t s) {
  using L = SL<QT, SWIGLU, WAVES, NC>;
  static_assert(L::LDS + 16 * L::ENTRY * 4 <= LDS_BYTES, "LDS");
  const int64_t items = a.max_tiles * ((a.N + L::RBW - 1) / L::RBW);
  if (items <= 0) return ARTLITE_OK;
  static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(k_stream<QT, SWIGLU, WAVES, NC>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
  const int cus = device_cus();
  if (!ok || cus <= 0) return fail(ARTLITE_EHIP, "streamed tiles: kernel set-up failed");
  int64_t grid = 0, entries = 0;
  const bool fits = stream_grid<QT, SWIGLU, WAVES, NC>(items, cus, grid, entries);
  if (dry) return fits ? ARTLITE_OK : ARTLITE_EINVAL;
  if (!fits) return fail(ARTLITE_EINVAL, "streamed tiles: %lld work items", (long long)items);
  k_stream<QT, SWIGLU, WAVES, NC><<<unsigned(grid), L::THREADS, L::LDS + size_t(entries) * L::ENTRY * 4, s>>>(a);
  ART_HIP(hipGetLastError());
  return ARTLITE_OK;
}

// (4 waves a workgroup; 8 where the slots then leave one workgroup of 4 a CU: Q6_K's tiles of 32 rows, whose down at 32
// rows an expert took 110 us with 4 and 93 with 8. Tiles of 64 rows in the formats they were measured in; Q6_K's slots
// would not fit them in LDS.)
template <int QT, int NC>
int launch_bm(const StreamArgs& a, bool dry, hipStream_t s) {
  constexpr int W = 2 * (SL<QT, true, 4, NC>::LDS + 2048) <= LDS_BYTES ? 4 : 8;
  if constexpr (NC == 4 && QT != ARTLITE_Q4_0 && QT != ARTLITE_Q4_K && QT != ARTLITE_Q8_0)
    return dry ? ARTLITE_EINVAL : fail(ARTLITE_EINVAL, "streamed tiles: %d rows of weight type %d", 16 * NC, QT);
  else
    return a.w[1] ? launch_t<QT, true, W, NC>(a, dry, s) : launch_t<QT, false, W, NC>(a, dry, s);
}

}  // namespace

bool stream_supported(int qtype, int K, int N) {
  const bool b32 = qtype == ARTLITE_Q4_0 || qtype == ARTLITE_Q8_0 || qtype == ARTLITE_Q4_1 || qtype == ARTLITE_IQ4_NL;
  const bool k256 = qtype == ARTLITE_Q4_K || qtype == ARTLITE_Q5_K || qtype == ARTLITE_Q6_K || qtype == ARTLITE_IQ4_XS ||
                    qtype == ARTLITE_Q3_K;
  return (b32 || k256) && K > 0 && K % (k256 ? 256 : 64) == 0 && N > 0;
}

#define ART_ST_QTYPES(X)                       \
  switch (a.qtype) {                           \
    case ARTLITE_Q4_0: X(ARTLITE_Q4_0);        \
    case ARTLITE_Q4_1: X(ARTLITE_Q4_1);        \
    case ARTLITE_Q8_0: X(ARTLITE_Q8_0);        \
    case ARTLITE_Q3_K: X(ARTLITE_Q3_K);        \
    case ARTLITE_Q4_K: X(ARTLITE_Q4_K);        \
    case ARTLITE_Q5_K: X(ARTLITE_Q5_K);        \
    case ARTLITE_Q6_K: X(ARTLITE_Q6_K);        \
    case ARTLITE_IQ4_NL: X(ARTLITE_IQ4_NL);    \
    default: X(ARTLITE_IQ4_XS);                \
  }

namespace {
// (dry: whether a launch takes the items, as a status and no message)
int by_type(const StreamArgs& a, bool dry, hipStream_t s) {
#define ART_ST(QT) \
  return a.bm == 16   ? launch_bm<QT, 1>(a, dry, s)  \
         : a.bm == 32 ? launch_bm<QT, 2>(a, dry, s) \
                      : launch_bm<QT, 4>(a, dry, s)
  ART_ST_QTYPES(ART_ST)
#undef ART_ST
}
}  // namespace

bool stream_fits(int qtype, bool swiglu, int N, int bm, int64_t max_tiles) {
  StreamArgs a{};
  static const uint8_t up = 0;
  a.w[1] = swiglu ? &up : nullptr;  // (a dry run: the kind alone)
  a.qtype = qtype;
  a.N = N;
  a.bm = bm;
  a.max_tiles = max_tiles;
  return by_type(a, true, nullptr) == ARTLITE_OK;
}

int launch_stream(const StreamArgs& a, hipStream_t s) {
  const bool swiglu = a.w[1] != nullptr;
  if (!stream_supported(a.qtype, a.K, a.N))
    return fail(ARTLITE_EINVAL, "streamed tiles: weight type %d, K %d, N %d", a.qtype, a.K, a.N);
  if (!a.w[0] || !a.a || !a.row_scale || (swiglu ? !a.h : !a.y16) || !a.tiles || !a.n_tiles || a.rows < 0 ||
      (a.bm != 16 && a.bm != 32 && a.bm != 64))
    return fail(ARTLITE_EINVAL, "streamed tiles: null or mismatched argument");
  if (int64_t(a.rows) * a.K * 2 >= (int64_t(1) << 32))
    return fail(ARTLITE_EINVAL, "streamed tiles: %d rows of %d beyond 32-bit offsets", a.rows, a.K);
  return by_type(a, false, s);
}

namespace {
template <int QT, bool SWIGLU>
int launch_few(const StreamFewArgs& a, hipStream_t s) {
  constexpr int RBW = SL<QT, SWIGLU, 1, 1>::RBW;
  const dim3 grid(unsigned((a.N + RBW - 1) / RBW), unsigned((a.rows + 15) / 16));
  if (a.a_lo)
    k_stream_few<QT, SWIGLU, 2><<<grid, 512, 0, s>>>(a);
  else
    k_stream_few<QT, SWIGLU, 1><<<grid, 512, 0, s>>>(a);
  ART_HIP(hipGetLastError());
  return ARTLITE_OK;
}
}  // namespace

int launch_stream_few(const StreamFewArgs& a, hipStream_t s) {
  const bool swiglu = a.w[1] != nullptr;
  if (!stream_supported(a.qtype, a.K, a.N))
    return fail(ARTLITE_EINVAL, "streamed dense rows: weight type %d, K %d, N %d", a.qtype, a.K, a.N);
  if (!a.w[0] || !a.a || (swiglu ? !a.h_hi || !a.h_lo : !a.y) || a.rows < 0 || a.rows > STREAM_FEW_ROWS)
    return fail(ARTLITE_EINVAL, "streamed dense rows: null or mismatched argument");
  if (a.rows == 0) return ARTLITE_OK;
#define ART_ST(QT) return swiglu ? launch_few<QT, true>(a, s) : launch_few<QT, false>(a, s)
  ART_ST_QTYPES(ART_ST)
#undef ART_ST
}
#undef ART_ST_QTYPES

}  // namespace artlite
