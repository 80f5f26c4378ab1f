// Prefill dequant GEMM for many rows (int4 and int8 weights): C =
// epi(A . deq(W)^T) on v_mfma_f32_32x32x16_f16, fp32 accumulation, one
// rounding.  Tiles of 32*MB rows by 256 weight rows, MB = 8, 4 or 2.
//
// Replaces dequant_matmul_int4_fp16 / dequant_matmul_int8_fp16
// (shaders/matmul_dequant_kernel.metal:55-223, :351-479; dispatched at
// src/ops/matmul.mm:1011-1021), with the fused epilogues of
// shaders/matmul_fused_epilogue.metal:97-124 and the SwiGLU of
// shaders/fused_swiglu.metal:48-84.
//
// Structure:
//  * Workgroup = 4 waves, one per SIMD, side by side along N: every wave
//    takes 64 weight rows (two blocks of 32; with SwiGLU 32 gate rows and
//    their 32 up rows) and all rows of the tile, over all of K.  A weight is
//    loaded and dequantized once per workgroup, in registers; activations
//    are moved to LDS once per workgroup and read by the four waves.
//  * Activations: direct-to-LDS 16-byte loads of 64-k tiles into a ring of 4
//    shared slots, XOR-swizzled per row (conflict-free fragment reads).  One
//    barrier per K-tile: it stands before the tile's last k-step, when every
//    wave holds its last fragments of this tile (so the slot can be refilled
//    with tile t + 4) and its own loads of tile t + 1 have landed.
//  * Weights: lane (c, h) of a block holds row c's 32 k at 64t + 32h (one
//    16-byte load for int4, two for int8), k-step s taking the 8 k at 8s; the
//    activation fragment of the same lane reads the same k.  A register ring
//    of 4 K-tiles.
//  * Scales and zeros: per wave, an LDS table of its 64 rows x the eight 32-k
//    pieces of four K-tiles, two of them in turn, filled two iterations ahead
//    by ordinary loads -- any number of groups, with no limit from LDS.
//  * The weights are the MFMA's first operand, so a lane's accumulator holds
//    four adjacent output columns of one row; the epilogue goes through a
//    per-wave LDS stage, 32 rows at a time, to 16-byte stores.
//
// Dequantization without forming q - 8 first, as fast_dq of mq_device.hpp (where
// its rounding is shown) but in natural k order, 4 instead of 5 VALU ops per
// pair of weights; int8 takes u = q + 128 as u * 2^-24.  It holds for scales of
// 2^-14 <= |s| < 4; a wave that meets another one takes the direct form for
// those K-tiles.
//
// What it measures (M = 4096, K = 3584, N = 37888, int4 g = 128 with SwiGLU):
// 1.05 ms, 1058 TFLOP/s, against 2.51 ms for the 64-column tiles of
// mq_gemmw.hip; plain fp16 weights in the vendor library: 0.90 ms.  With all
// CUs running the clock drops to 1.76 GHz and the matrix cores are busy 54 % of
// its cycles (counters); the same loop with nothing but its MFMAs takes 0.79
// ms, which is all of the cycles at 1.3 GHz.  Taking one thing out of the loop
// at 18 workgroups (1.28 us a K-tile, full clock; variants, not kept): dequant
// 1.24, activation loads 1.12, fragment reads 1.27, weight loads 1.21, all four
// 1.05; spreading the activation loads over the k-steps took it to 1.21.
// 256 rows by 64 columns per wave keep the dequant at two VALU ops per
// MFMA and LDS reads at 5/8 of its rate.  128-row tiles (two workgroups per
// CU) dequantize twice as often and are within 3 % at full load; they fill
// the CUs where there are fewer rows.
//
// Hazards of the inline-asm MFMAs (the compiler does not see inside them):
// their weight operands are written at least two MFMAs before the first use,
// activation fragments by LDS reads that the compiler waits for; accumulators
// are only touched by MFMAs until the read-out, after 24 wait states.
#include "mq_device.hpp"
#include "mq_launch.hpp"

#include <algorithm>
#include <type_traits>

namespace mq {
namespace {

constexpr int GN_ROWS = 256;   // weight rows per workgroup (64 per wave)
constexpr int GN_NS = 4;       // activation slots = K-tiles per loop iteration

struct GNArgs {
  const _Float16* A; int64_t lda;
  const unsigned char* W; int64_t ldw;
  const _Float16* scales; const _Float16* zeros;
  EpiArgs ep;
  _Float16* C; int64_t ldc;
  int M, N, K, G, gshift;
  int F;                // output columns: N/2 with SwiGLU, else N
  int nbm, nbn, KT, xcd;
  int KP, ktp;          // K parts, K-tiles per part (the last may have fewer)
  float* part;          // [KP][M][ldp] fp32 partial sums (KP > 1)
  int ldp, up0;         // row stride, first up column (SwiGLU)
  int gm;               // M blocks per group of the tile order
  int vec_store;        // C rows 16-byte aligned
  int vec_resid;        // residual rows 16-byte aligned
  uint32_t a_bytes, w_bytes, s_bytes, z_bytes;
};

__device__ __forceinline__ void gn_dma16(rsrc_t r, u4* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

// Activation slot I: a separate LDS array per slot, so that the compiler's
// load-counter waits tell one slot's loads from another's.
template <int I, int S>
__device__ __forceinline__ u4 (&gn_slot())[S] {
  __shared__ u4 a[S];
  return a;
}

template <int FMT, int MB, bool SWI, bool KS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MB == 8 ? 1 : 2, MB == 8 ? 1 : 2))) void
gemmn_kernel(GNArgs p) {
  constexpr int BM = 32 * MB;                   // rows per tile
  constexpr int BNO = SWI ? 128 : 256;          // output columns per tile
  constexpr int WCO = SWI ? 32 : 64;            // output columns per wave
  constexpr int SLOTU = BM * 8;                 // 16-byte pieces per activation slot
  constexpr int ND = BM / 32;                   // DMA instructions per wave and K-tile (8 rows each)
  constexpr int NW = FMT == FMT_INT4 ? 2 : 4;   // weight loads per wave and K-tile
  constexpr int NL = NW / 2;                    // weight loads per block
  constexpr int NM = 2 * MB;                    // MFMAs per k-step
  constexpr int DQ = (ND + 3) / 4;              // DMA instructions per k-step, at most
  // weight ring depth in K-tiles: 4, or 2 where registers are short
  constexpr int WD = FMT == FMT_INT8 && MB < 8 ? 2 : 4;
  // scale | zero << 16, [wave][iteration & 1][piece e][column ^ 8e]
  __shared__ uint32_t lds_sz[4][2][8 * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  int id = blockIdx.x, kp = 0;
  if (p.xcd) {   // workgroup i runs on XCD i % 8: give each XCD a contiguous run of tiles
    const int per = gridDim.x >> 3;
    id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  }
  if constexpr (KS) {   // parts of one K range together
    const int tiles = p.nbm * p.nbn;
    kp = id / tiles;
    id -= kp * tiles;
  }
  // groups of gm M blocks by all N blocks, M fastest: the tiles that run at
  // one time on an XCD form a compact rectangle and share its L2
  const int per = p.gm * p.nbn;
  const int grp = id / per, inside = id - grp * per;
  const int gmh = min(p.gm, p.nbm - grp * p.gm);
  const int nb = inside / gmh, mb = grp * p.gm + (inside - nb * gmh);
  const int m0 = mb * BM, n0 = nb * BNO;
  // this part's K range: operands from its first k on
  const int kt0 = KS ? kp * p.ktp : 0;
  const int KT = KS ? min(p.ktp, p.KT - kt0) : p.KT;
  const int kbase = 64 * kt0, klen = min(p.K - kbase, 64 * KT);
  constexpr int WTB = FMT == FMT_INT4 ? 32 : 64;   // bytes of a weight row per K-tile
  const rsrc_t ar = make_rsrc(p.A + kbase, p.a_bytes - (uint32_t)kbase * 2u);
  const rsrc_t wr = make_rsrc(p.W + kt0 * WTB, p.w_bytes - (uint32_t)(kt0 * WTB));
  const rsrc_t sr = make_rsrc(p.scales, p.s_bytes);
  const rsrc_t zr = make_rsrc(p.zeros, p.z_bytes);

  // ---- activations: DMA instruction i of wave w moves rows 8(ND w + i)..+7;
  // lane l -> row l/8 of them, LDS position l%8, k-piece (l%8) ^ (row%8) ----
  const int pa = (lane & 7) ^ (lane >> 3);
  const uint32_t adma = (uint32_t)((m0 + 8 * ND * w + (lane >> 3)) * p.lda * 2) + 16u * pa;
  // the last K-tile of a K that ends inside it: its upper half reads zeros
  const uint32_t adma_tail = (klen & 63) && pa >= 4 ? kOob : adma;
  const uint32_t rstride = (uint32_t)(8 * p.lda * 2);
  auto slot = [&](auto ic) -> u4* { return gn_slot<decltype(ic)::value, SLOTU>(); };
  // K-tiles past the end: an offset past every range (reads zeros)
  auto dma_one = [&](int t, u4* sl, int i) {
    const uint32_t so = t >= KT ? kOob : (uint32_t)t * 128u;
    gn_dma16(ar, sl + 64 * (ND * w + i), t == KT - 1 ? adma_tail : adma, so + i * rstride);
  };
  // fragment of row block i, k-step s: row 32i + c, k-piece 4h + s (bytes;
  // opaque to the compiler, which else keeps one address per slot and step)
  uint32_t ard[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    ard[s] = (uint32_t)(c * 8 + ((4 * h + s) ^ (c & 7))) * 16u;
    asm volatile("" : "+v"(ard[s]));
  }
  auto frag = [&](const u4* sl, uint32_t off, int i) -> h8 {
    return __builtin_bit_cast(h8, *(const u4*)((const char*)sl + off + 4096 * i));
  };

  // ---- weights: block j, lane c ----
  uint32_t woff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int o = n0 + WCO * w + (SWI ? 0 : 32 * j) + c;
    const int row = SWI && j ? p.F + o : o;
    woff[j] = o < p.F ? (uint32_t)(row * p.ldw) + (uint32_t)(16 * NL * h) : kOob;
  }
  u4 wring[WD][2][NL];
  auto load_w = [&](int t, u4 (&dst)[2][NL]) {
    const uint32_t so = t >= KT ? 0u : (uint32_t)(t * WTB);   // past the end: any finite weights
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < NL; ++u)
        dst[j][u] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(wr, woff[j] + 16u * u, so, 0));
  };

  // ---- scale | zero table: load r covers columns 8r..8r+7 (lane / 8) of the
  // wave, piece e = lane % 8 of the iteration's 256 k ----
  const int te = lane & 7, tc = lane >> 3;
  const uint32_t tbase = (uint32_t)((n0 + WCO * w + tc) * (int64_t)p.G * 2);
  // half a table at a time (4 columns of 8 pieces per lane): 8 registers
  uint32_t ts[4], tz[4];
  auto tab_off = [&](int it) {
    const int k = kbase + 256 * it + 32 * te;
    return tbase + 2u * (uint32_t)(p.gshift >= 31 ? 0 : min(k >> p.gshift, p.G - 1));
  };
  auto tab_load = [&](uint32_t off, int half, int r) {
    const uint32_t so = (uint32_t)(((SWI ? half * p.F : 32 * half) + 8 * r) * (int64_t)p.G * 2);
    ts[r] = __builtin_amdgcn_raw_buffer_load_b16(sr, off, so, 0);
    tz[r] = __builtin_amdgcn_raw_buffer_load_b16(zr, off, so, 0);
  };
  // column 32 half + 8r + tc, piece te: dword te * 64 + (column ^ 8 te), as
  // one XOR of a lane part and a constant
  uint32_t tlane = (uint32_t)(w * 1024 + te * 72 + tc) * 4u;
  // columns that exist: 32 half + 8r below tl (SwiGLU: 8r, of each half)
  int tl = p.F - (n0 + WCO * w) - tc;
  auto tab_write = [&](int it, int half, int r) -> bool {
    asm volatile("" : "+v"(tlane), "+v"(tl));   // not hoisted out of the loop
    const uint32_t off = (tlane ^ (uint32_t)(4 * (32 * half + 8 * r))) + (it & 1) * 2048u;
    *(uint32_t*)((char*)lds_sz + off) = (ts[r] & 0xFFFFu) | (tz[r] << 16);
    // not of the fast form's range (columns past the end: whatever)
    return ((ts[r] >> 10) & 31u) - 1u >= 16u && (SWI ? 8 * r : 32 * half + 8 * r) < tl;
  };

  f16v acc[MB][2];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f16v){};

  // dequant constants
  const uint32_t nmask = 0x00F0000Fu;
  const uint32_t sel0 = 0x0c000c00u, sel1 = 0x0c010c01u, sel2 = 0x0c020c02u, sel3 = 0x0c030c03u;
  const uint32_t z8lo = 0x0c010c00u, z8hi = 0x0c030c02u;     // int8: bytes 0,1 / 2,3 under 0

  // per block of a K-tile: e = s | z << 16; S, C = the
  // addend pair, PP = the power-of-two pair of the fast form
  struct Dq { uint32_t e, S, C, PP; };
  auto derive = [&](uint32_t e, Dq& d) {
    d.e = e;
    const uint32_t se = FMT == FMT_INT4 ? 25u << 10 : 29u << 10;
    d.S = (e & 0xFFFF83FFu) | se;
    const h2 s2 = __builtin_shufflevector(as_h2(d.S), as_h2(d.S), 0, 0);
    d.C = as_u32(s2 * as_h2(FMT == FMT_INT4 ? 0x80808008u : 0x80808080u));   // -2^-21 | -2^-17
    const uint32_t ee = __builtin_amdgcn_perm(0u, e, 0x01000100u) & 0x7C007C00u;
    d.PP = ee + (FMT == FMT_INT4 ? 0x28003800u : 0x28002800u);
  };

  // op n of the dequant of one block's 8 weights (4 registers x)
  constexpr int NO = FMT == FMT_INT4 ? 16 : 14;
  auto dq_op = [&](int n, const u4 (&wt)[NL], int s, const Dq& d, uint32_t (&x)[4], uint32_t (&u)[2]) {
    const int m = FMT == FMT_INT4 ? n : n - 2, i = m & 3;
    if constexpr (FMT == FMT_INT4) {
      // a byte into both halves, then its low nibble there, its high nibble here
      const uint32_t sel = i == 0 ? sel0 : i == 1 ? sel1 : i == 2 ? sel2 : sel3;
      if (n < 4) asm volatile("v_perm_b32 %0, 0, %1, %2" : "=v"(x[i]) : "v"(wt[0][s]), "s"(sel));
      else if (n < 8) asm volatile("v_and_b32 %0, %1, %0" : "+v"(x[i]) : "s"(nmask));
    } else {
      // q + 128, one byte to each half
      if (n < 2) asm volatile("v_xor_b32 %0, 0x80808080, %1" : "=v"(u[n]) : "v"(wt[s >> 1][2 * (s & 1) + n]));
      else if (m < 4) asm volatile("v_perm_b32 %0, 0, %1, %2" : "=v"(x[i]) : "v"(u[i >> 1]), "s"((i & 1) ? z8hi : z8lo));
    }
    constexpr int F1 = FMT == FMT_INT4 ? 8 : 4;
    if (m >= F1 && m < F1 + 4)
      asm volatile("v_pk_fma_f16 %0, %0, %1, %2 op_sel_hi:[1,0,1]" : "+v"(x[i]) : "v"(d.S), "v"(d.C));
    else if (m >= F1 + 4)
      asm volatile("v_pk_fma_f16 %0, %0, %1, %2 op_sel:[0,0,1] op_sel_hi:[1,1,1] neg_lo:[0,0,1] neg_hi:[0,0,1]"
                   : "+v"(x[i]) : "v"(d.PP), "v"(d.e));
  };
  auto any_lane = [](bool b) -> uint32_t {
    const uint64_t m = __builtin_amdgcn_ballot_w64(b);
    return __builtin_amdgcn_readfirstlane((uint32_t)m | (uint32_t)(m >> 32));
  };
  // the direct form (any scale); in asm so that its constants stay in SGPRs
  const uint32_t nib_m = 0x2C003C00u, nib_a = 0xD480E408u;   // (1, 1/16), (-1032, -72)
  const uint32_t m1152 = 0xE480E480u, magic = 0x64006400u;
  auto dq_direct = [&](const u4 (&wt)[NL], int s, uint32_t e) -> h8 {
    uint32_t x[4];
#define GN_ALL _Pragma("unroll") for (int i = 0; i < 4; ++i)
    if constexpr (FMT == FMT_INT4) {
      GN_ALL asm volatile("v_perm_b32 %0, 0, %1, %2" : "=v"(x[i]) : "v"(wt[0][s]), "s"(i == 0 ? sel0 : i == 1 ? sel1 : i == 2 ? sel2 : sel3));
      GN_ALL asm volatile("v_and_b32 %0, %1, %0" : "+v"(x[i]) : "s"(nmask));
      GN_ALL asm volatile("v_or_b32 %0, %1, %0" : "+v"(x[i]) : "s"(magic));
      GN_ALL asm volatile("v_pk_mul_f16 %0, %0, %1" : "+v"(x[i]) : "s"(nib_m));   // 1024 + lo, 64 + hi
      GN_ALL asm volatile("v_pk_add_f16 %0, %0, %1" : "+v"(x[i]) : "s"(nib_a));
    } else {
      GN_ALL asm volatile("v_xor_b32 %0, 0x80808080, %1" : "=v"(x[i]) : "v"(wt[s >> 1][2 * (s & 1) + (i >> 1)]));
      GN_ALL asm volatile("v_perm_b32 %0, 0, %0, %1" : "+v"(x[i]) : "s"((i & 1) ? z8hi : z8lo));
      GN_ALL asm volatile("v_or_b32 %0, %1, %0" : "+v"(x[i]) : "s"(magic));
      GN_ALL asm volatile("v_pk_add_f16 %0, %0, %1" : "+v"(x[i]) : "s"(m1152));
    }
    GN_ALL asm volatile("v_pk_mul_f16 %0, %0, %1 op_sel_hi:[1,0]" : "+v"(x[i]) : "v"(e));
    GN_ALL asm volatile("v_pk_add_f16 %0, %0, %1 op_sel:[0,1] neg_lo:[0,1] neg_hi:[0,1]" : "+v"(x[i]) : "v"(e));
#undef GN_ALL
    u4 o = (u4){x[0], x[1], x[2], x[3]};
    asm volatile("s_nop 3" : "+v"(o));
    return __builtin_bit_cast(h8, o);
  };

  uint32_t bad0 = 0, bad1 = 0;   // a scale of iteration it / it + 1 needs the direct form
  // One k-step: the 2 MB MFMAs of (bq, af), after each of them a share of the
  // dequant ops of the next k-step's two blocks, one of the next k-step's
  // fragment reads after every second, and `extra(m)`.
  // EARLY: the reads come one after every MFMA, done by the middle.  `ne`: s | z << 16
  // of the direct form (`extra` may set nd to the next K-tile's once it is used).
  auto step = [&](auto earlyc, const h8 (&af)[MB], const h8 (&bq)[2], const u4* nsl, uint32_t nard, h8 (&naf)[MB],
                  const u4 (&nwt)[2][NL], int ns, const Dq (&nd)[2], h8 (&nbq)[2], auto extra) {
    constexpr bool EARLY = decltype(earlyc)::value;
    const uint32_t ne[2] = {nd[0].e, nd[1].e};
    uint32_t x[2][4], u[2][2];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int i = m >> 1, j = m & 1;
      asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bq[j]), "v"(af[i]));
      if (EARLY ? m < MB : j == 0) naf[EARLY ? m : i] = frag(nsl, nard, EARLY ? m : i);
#pragma unroll
      for (int o = 0; o < 2 * NO; ++o)   // every op done two MFMAs before the step's end
        if (m < NM - 2 && o >= m * 2 * NO / (NM - 2) && o < (m + 1) * 2 * NO / (NM - 2))
          dq_op(o % NO, nwt[o / NO], ns, nd[o / NO], x[o / NO], u[o / NO]);
      extra(m);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u4 o;
      o.x = x[j][0]; o.y = x[j][1]; o.z = x[j][2]; o.w = x[j][3];
      nbq[j] = __builtin_bit_cast(h8, o);
    }
    // the iteration's own scales, or the next one's (whose first k-step is
    // made here)
    if (bad0 | bad1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        nbq[j] = dq_direct(nwt[j], ns, ne[j]);
      }
    }
  };

  // ---- prologue ----
  {
    const uint32_t off = tab_off(0);
    bool bad = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) tab_load(off, 0, r);
    uint32_t us[4], uz[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) { us[r] = ts[r]; uz[r] = tz[r]; tab_load(off, 1, r); }
    auto first = [&](auto ic) {
      constexpr int I = decltype(ic)::value;
#pragma unroll
      for (int i = 0; i < (I < 3 ? ND : DQ); ++i) dma_one(I, slot(ic), i);   // (tile 3: the rest in the loop)
      if (I < WD) load_w(I, wring[I % WD]);
    };
    first(std::integral_constant<int, 0>{});
    first(std::integral_constant<int, 1>{});
    first(std::integral_constant<int, 2>{});
    first(std::integral_constant<int, 3>{});
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= tab_write(0, 1, r);
#pragma unroll
    for (int r = 0; r < 4; ++r) { ts[r] = us[r]; tz[r] = uz[r]; bad |= tab_write(0, 0, r); }
    bad0 = any_lane(bad);
  }

  // the wave's own loads of the tile that is read next have landed: those
  // issued after them are two tiles' activations and at least two tiles'
  // weights; at tiles 0 and 1 of a 2-deep weight ring one tile's weights and
  // the eight scale and zero loads of tile 0 (NW = 4 of them are needed)
  auto tile_ready = [&]() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * ND + 2 * NW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * ND + DQ + (WD - 1) * NW) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  h8 afA[MB], afB[MB], bqA[2], bqB[2];
  Dq dq[2];
  // entry of tile R, block j: piece e = 2R + h, dword e * 64 + ((32 j + c) ^ 8 e)
  uint32_t rlane[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    rlane[o] = (uint32_t)(w * 1024 + 64 * h + (c ^ (8 * h) ^ (16 * o))) * 4u;
    asm volatile("" : "+v"(rlane[o]));
  }
  auto read_sz = [&](int it, int R, int j) -> uint32_t {
    return *(const uint32_t*)((const char*)lds_sz + rlane[R & 1] + (it & 1) * 2048u + 4u * (128 * R + 32 * (j ^ (R >> 1))));
  };
#pragma unroll
  for (int i = 0; i < MB; ++i) afA[i] = frag(slot(std::integral_constant<int, 0>{}), ard[0], i);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    derive(read_sz(0, 0, j), dq[j]);
    bqA[j] = dq_direct(wring[0][j], 0, dq[j].e);
  }

  // K-tile t = 4 it + R: activations in slot R, weights in ring slot R % WD.
  // The next iteration's table goes into the other table slot, half by half:
  // loaded at (tile, k-step) (0, 0) and (1, 3), written at (1, 2) and (3, 0).
  bool tbad = false;
  auto tile = [&](auto rc, int it) {
    constexpr int R = decltype(rc)::value, RN = (R + 1) & 3;
    const int t = 4 * it + R;
    u4* const cur = slot(std::integral_constant<int, R>{});
    u4* const nxt = slot(std::integral_constant<int, RN>{});
    uint32_t toff = 0, e2[2];
    if constexpr (R == 0 || R == 1) toff = tab_off(it + 1);
    // the slot that the barrier of tile t - 1 freed: a quarter of its refill
    // (K-tile t + 3) per k-step, so that the four waves' loads spread out
    auto refill = [&](int tt, u4* sl, int q, int m) {
#pragma unroll
      for (int i = 0; i < ND; ++i)
        if (i * 4 / ND == q && 2 + (i % DQ) * NM / DQ == m) dma_one(tt, sl, i);
    };
    u4* const prv = slot(std::integral_constant<int, (R + 3) & 3>{});
    constexpr auto late = std::false_type{};
    step(late, afA, bqA, cur, ard[1], afB, wring[R % WD], 1, dq, bqB, [&](int m) {
      refill(t + 3, prv, 1, m);
      if (R == 0 && m < 4) tab_load(toff, 0, m);
      if (R == 3 && m < 4) tbad |= tab_write(it + 1, 1, m);
    });
    step(late, afB, bqB, cur, ard[2], afA, wring[R % WD], 2, dq, bqA, [&](int m) {
      refill(t + 3, prv, 2, m);
      if (m < 2) e2[m] = read_sz(R == 3 ? it + 1 : it, RN, m);
    });
    step(std::true_type{}, afA, bqA, cur, ard[3], afB, wring[R % WD], 3, dq, bqB, [&](int m) {
      refill(t + 3, prv, 3, m);
      if (R == 1 && m < 4) tbad |= tab_write(it + 1, 0, m);
      if (m >= NM - 2) derive(e2[m - (NM - 2)], dq[m - (NM - 2)]);   // K-tile t + 1 (dq's last use is behind)
    });
    if constexpr (R == 3) {
      bad1 = any_lane(tbad);
      tbad = false;
    }
    // every wave holds its last fragments of this tile, and tile t + 1 is in LDS
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    tile_ready();
    step(late, afB, bqB, nxt, ard[0], afA, wring[RN % WD], 0, dq, bqA, [&](int m) {
      refill(t + 4, cur, 0, m);
      if (R == 1 && m < 4) tab_load(toff, 1, m);
      if (m == NM - 1) load_w(t + WD, wring[R % WD]);
    });
    if constexpr (R == 3) {
      bad0 = bad1;
      bad1 = 0;
    }
  };
  // one exit: leaving the loop between tiles makes the compiler copy (and
  // spill) the accumulators
  int it = 0;
  do {
    tile(std::integral_constant<int, 0>{}, it);
    if (4 * it + 1 < KT) {
      tile(std::integral_constant<int, 1>{}, it);
      if (4 * it + 2 < KT) {
        tile(std::integral_constant<int, 2>{}, it);
        if (4 * it + 3 < KT) tile(std::integral_constant<int, 3>{}, it);
      }
    }
    ++it;
  } while (4 * it < KT);

  // ---- epilogue ----
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");   // MFMA results retired
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load into a slot is in flight
  __syncthreads();                                   // no wave reads one any more
  // Wave w stages NBS row blocks at a time in slot w: fp32 rows of PR 16-byte
  // pieces, piece p of row r at p ^ (r % 8) (conflict-free both ways), read
  // back a row per group of lanes.  One wave's LDS accesses complete in
  // order: no barrier.  The read-back is a loop: unrolled over the row blocks
  // the epilogue was 30 KiB of code that each workgroup runs once, and its
  // instruction fetches cost up to 40 us a launch.
  constexpr int SC = KS ? 64 : WCO;   // staged columns (K parts with SwiGLU: gate, then up)
  constexpr int PR = SC / 4;
  constexpr int NBS = SLOTU / (32 * PR) < MB ? SLOTU / (32 * PR) : MB;
  f4* const stg = (f4*)(w == 0 ? slot(std::integral_constant<int, 0>{})
                        : w == 1 ? slot(std::integral_constant<int, 1>{})
                        : w == 2 ? slot(std::integral_constant<int, 2>{})
                                 : slot(std::integral_constant<int, 3>{}));
  constexpr int PPR = SC / 8;        // 8-column pieces per row
  constexpr int RPP = 64 / PPR;      // rows per pass of the wave
  const int cp = lane % PPR, cc = 8 * cp, rr = lane / PPR;
  const bool upc = KS && SWI && cc >= 32;                       // an up column of a K part
  const int col = n0 + WCO * w + (upc ? cc - 32 : cc);
  const int nc = min(8, p.F - col);  // columns of this lane's piece (<= 0: none)
  const int kind = SWI || KS ? (int)EPI_NONE : p.ep.epi;
  f4 bias[2] = {(f4){0.f, 0.f, 0.f, 0.f}, (f4){0.f, 0.f, 0.f, 0.f}};   // of this lane's columns
  if (epi_needs_bias(kind)) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < nc) bias[e >> 2][e & 3] = (float)((const _Float16*)p.ep.bias)[col + e];
  }
#pragma unroll
  for (int b0 = 0; b0 < MB; b0 += NBS) {
#pragma unroll
    for (int i = 0; i < NBS; ++i)
#pragma unroll
      for (int vg = 0; vg < 4; ++vg) {
        f4* const b = stg + (32 * i + c) * PR;
        if constexpr (SWI && !KS) {
          f4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = silu_f32((float)(_Float16)acc[b0 + i][0][4 * vg + e]) * (float)(_Float16)acc[b0 + i][1][4 * vg + e];
          b[(2 * vg + h) ^ (c & 7)] = v;
        } else {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            f4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[b0 + i][j][4 * vg + e];
            b[(8 * j + 2 * vg + h) ^ (c & 7)] = v;
          }
        }
      }
    const int rend = nc <= 0 ? 0 : min(32 * NBS, p.M - (m0 + 32 * b0));
#pragma unroll 1
    for (int r = rr; r < rend; r += RPP) {
      const int64_t row = m0 + 32 * b0 + r;
      f4 v0 = stg[r * PR + ((2 * cp) ^ (r & 7))], v1 = stg[r * PR + ((2 * cp + 1) ^ (r & 7))];
      if constexpr (KS) {   // rows of ldp columns, a multiple of 8: whole pieces
        f4* const dst = (f4*)(p.part + ((int64_t)kp * p.M + row) * p.ldp + (upc ? p.up0 : 0) + col);
        dst[0] = v0;
        dst[1] = v1;
      } else {
        if (kind == EPI_RESIDUAL) {
          const _Float16* rp = (const _Float16*)p.ep.resid + row * p.ep.ldr + col;
          if (p.vec_resid && nc == 8) {
            const h8 rv = *(const h8*)rp;
#pragma unroll
            for (int e = 0; e < 4; ++e) { v0[e] += (float)rv[e]; v1[e] += (float)rv[4 + e]; }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (e < nc) {
                if (e < 4) v0[e & 3] += (float)rp[e];
                else v1[e & 3] += (float)rp[e];
              }
          }
        } else if (kind != EPI_NONE) {
          v0 += bias[0];
          v1 += bias[1];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (kind == EPI_BIAS_RELU) { v0[e] = fmaxf(v0[e], 0.0f); v1[e] = fmaxf(v1[e], 0.0f); }
            if (kind == EPI_BIAS_SILU) { v0[e] = silu_f32(v0[e]); v1[e] = silu_f32(v1[e]); }
          }
        }
        h8 hv;
#pragma unroll
        for (int e = 0; e < 4; ++e) { hv[e] = (_Float16)v0[e]; hv[4 + e] = (_Float16)v1[e]; }
        _Float16* dst = p.C + row * p.ldc + col;
        if (p.vec_store && nc == 8) {
          *(h8*)dst = hv;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < nc) dst[e] = hv[e];
        }
      }
    }
  }
}

// Sum of the K parts in part order (deterministic), epilogue, fp16 rows:
// 8 output columns per thread.
template <bool SWI>
__global__ __launch_bounds__(256) void gemmn_sum_kernel(GNArgs p) {
  const int ppr = (p.F + 7) >> 3;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int row = (int)(id / ppr), col = 8 * (int)(id - (int64_t)row * ppr);
  if (row >= p.M) return;
  const float* src = p.part + (int64_t)row * p.ldp + col;
  const int64_t ps = (int64_t)p.M * p.ldp;
  constexpr int NH = SWI ? 2 : 1;
  f4 v[NH][2] = {};
#pragma unroll 4
  for (int q = 0; q < p.KP; ++q)
#pragma unroll
    for (int u = 0; u < NH; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) v[u][e] += *(const f4*)(src + q * ps + u * p.up0 + 4 * e);
  const int nc = min(8, p.F - col);
  h8 hv;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float x = v[0][e >> 2][e & 3];
    if constexpr (SWI) x = silu_f32((float)(_Float16)x) * (float)(_Float16)v[NH - 1][e >> 2][e & 3];
    else if (p.ep.epi != EPI_NONE && e < nc) x = epi_apply(x, (int64_t)row, col + e, p.ep);
    hv[e] = (_Float16)x;
  }
  _Float16* dst = p.C + (int64_t)row * p.ldc + col;
  if (p.vec_store && nc == 8) *(h8*)dst = hv;
  else
    for (int e = 0; e < nc; ++e) dst[e] = hv[e];
}

template <int FMT, int MB>
hipError_t launch_mb(const GNArgs& k, bool swi, int nwg, hipStream_t s) {
  const dim3 g(nwg), b(256);
  if (k.KP > 1) {
    if (swi) hipLaunchKernelGGL((gemmn_kernel<FMT, MB, true, true>), g, b, 0, s, k);
    else hipLaunchKernelGGL((gemmn_kernel<FMT, MB, false, true>), g, b, 0, s, k);
    const dim3 gs((unsigned)(((int64_t)k.M * ((k.F + 7) / 8) + 255) / 256));
    if (swi) hipLaunchKernelGGL((gemmn_sum_kernel<true>), gs, b, 0, s, k);
    else hipLaunchKernelGGL((gemmn_sum_kernel<false>), gs, b, 0, s, k);
  } else {
    if (swi) hipLaunchKernelGGL((gemmn_kernel<FMT, MB, true, false>), g, b, 0, s, k);
    else hipLaunchKernelGGL((gemmn_kernel<FMT, MB, false, false>), g, b, 0, s, k);
  }
  return hipGetLastError();
}

}  // namespace

bool gemmn_supported(const LinearArgs& a) {
  if (a.fmt != FMT_INT4 && a.fmt != FMT_INT8) return false;
  if (a.prenorm || a.M < 1 || a.N < 1 || a.K < 64 || a.K % 32 != 0) return false;
  if (a.epi == EPI_SWIGLU && a.F * 2 != a.N) return false;
  if (a.lda % 8 != 0 || ((uintptr_t)a.A & 15) != 0) return false;     // 16-byte activation pieces
  if (a.ldw % 16 != 0 || ((uintptr_t)a.W & 15) != 0) return false;    // 16-byte weight loads
  if (((uintptr_t)a.scales & 1) || ((uintptr_t)a.zeros & 1)) return false;
  const bool per_channel = a.G == 1;
  if (!per_channel && (a.g < 32 || (a.g & (a.g - 1)) != 0)) return false;   // a lane's 32 k in one group
  // 32-bit buffer offsets, with the rows a tile may reach past the end
  const int64_t lim = (int64_t)1 << 31;
  if (((int64_t)a.M + 256) * a.lda * 2 >= lim || ((int64_t)a.N + 256) * a.ldw >= lim) return false;
  return ((int64_t)a.N + 256) * a.G * 2 < lim;
}

namespace {

// the start of the per-stream workspace holds the other kernels' counters,
// which must stay zero
constexpr size_t kCntBytesN = 65536;

// Launch-time model (microseconds), per tile height, fitted to 21300 measured
// launches of 6000 drawn shapes (M = 17..4096, up to 640 with 64 rows; K =
// 512..18944, N = 512..37888, int4 and int8, all group sizes and epilogues, 1-64
// K parts): 7 % rms with 64 and 128 rows, 8 % with 256.
//  * 256 rows: one workgroup per CU.  A K-tile takes 1.20 us, and 1.35 when
//    all CUs run (the clock drops under the load).
//  * 128 and 64 rows: two workgroups fit a CU.  A K-tile takes 0.82-0.93 us
//    (128 rows) or 0.71-0.80 (64) alone, 1.94 or 1.36 in each of two.
//  * int8 takes 0.10-0.33 us more per K-tile: twice the weight loads, and
//    with 64 and 128 rows half the ring depth.
//  * K parts: their sums are written and read once, 0.2 us per MB, and a
//    thread adds all parts of its 8 columns, 0.16 us a part, or 0.5 with SwiGLU
//    (half the threads with twice the loads; where they are few, nothing hides
//    the loads' latency).
//  * The bytes of scales, outputs and residual; rows that are not 16-byte
//    aligned are written, and a residual read, element by element.
struct NFit {
  double launch, round, tile, load, i8;        // tile: a K-tile in a full CU
  double two, alone, alone_i8, alone_load;     // two workgroups per CU: a K-tile of the second, of one alone
  double scale_mb, out_mb, bias_mb, resid_mb, silu_mb, odd_mb, odd_resid_mb;
  double split, split_swi, part, part_swi, part_mb, split_i8;
};
constexpr NFit kFit64 = {9.38, -4.33, 1.359, 0.009, 0.327, 1.186, 0.713, 0.112, 0.122, 0.955, 0.044, 0.270, 0.413,
                         0.466, 0.683, 0.579, 1.56, -0.88, 0.156, 0.402, 0.229, 0.16};
constexpr NFit kFit128 = {11.88, -4.48, 1.940, 0.273, 0.254, 1.421, 0.820, 0.102, 0.140, 0.484, 0.194, 0.101, 0.312,
                          0.410, 0.571, 0.678, 0.28, -0.71, 0.160, 0.372, 0.210, 0.10};
constexpr NFit kFit256 = {9.78, 1.19, 1.206, 0.136, 0.103, 0.0, 0.0, 0.0, 0.0, 0.117, 0.383, 0.094, 0.454,
                          0.445, 0.575, 0.709, -1.80, -0.02, 0.172, 0.317, 0.205, 0.76};

double estimate(const LinearArgs& a, int mb, int64_t wgs, int KP, int ktp, double part_mb, int cus) {
  const NFit& f = mb == 8 ? kFit256 : mb == 4 ? kFit128 : kFit64;
  const bool swi = a.epi == EPI_SWIGLU;
  const double i8 = a.fmt == FMT_INT8 ? 1.0 : 0.0;
  const double out_mb = 2e-6 * a.M * (swi ? a.F : a.N);
  double t = f.launch + f.scale_mb * 4e-6 * a.N * a.G + f.out_mb * out_mb;
  if (mb == 8) {
    const double rounds = (double)wgs / cus, whole = std::ceil(rounds);
    const double tk = f.tile + f.i8 * i8 + f.load * 2.0 * std::max(0.0, std::min(1.0, rounds) - 0.5);
    t += (whole <= 3 ? whole : rounds + 0.5) * (f.round + ktp * tk);
  } else {
    const int64_t slots = 2 * (int64_t)cus, full = wgs / slots, rem = wgs - full * slots;
    t += full * (f.round + ktp * (f.tile + f.i8 * i8));
    if (rem > cus) t += f.round + ktp * (f.two + f.i8 * i8 + f.load * (double)(rem - cus) / cus);
    else if (rem > 0) t += f.round + ktp * (f.alone + f.alone_i8 * i8) * (1.0 + f.alone_load * (double)rem / cus);
  }
  if (a.epi == EPI_RESIDUAL) t += (f.resid_mb + (a.ldr % 8 ? f.odd_resid_mb : 0.0)) * out_mb;
  if (epi_needs_bias(a.epi)) t += (f.bias_mb + (a.epi == EPI_BIAS_SILU ? f.silu_mb : 0.0)) * out_mb;
  if (a.ldc % 8) t += f.odd_mb * out_mb;
  if (KP > 1) t += f.split + f.split_i8 * i8 + f.part_mb * part_mb + f.part * KP + (swi ? f.split_swi + f.part_swi * KP : 0.0);
  return t;
}

}  // namespace

GemmnPlan gemmn_plan(const LinearArgs& a, int cus, bool allow_split, int mb, int kp) {
  GemmnPlan best{};
  if (!gemmn_supported(a)) return best;
  const bool swi = a.epi == EPI_SWIGLU;
  const int F = swi ? a.F : a.N;
  const int KT = (a.K + 63) / 64;
  const int64_t ld = (int64_t)((F + 7) & ~7) * (swi ? 2 : 1);
  for (int m = 2; m <= 8; m *= 2) {
    if (mb ? m != mb : m == 2 && a.M > 640) continue;   // (64 rows: on 676 shapes from 321 to 640 the fastest height on 255; not measured beyond)
    const int64_t tiles = (int64_t)((a.M + 32 * m - 1) / (32 * m)) * ((F + (swi ? 127 : 255)) / (swi ? 128 : 256));
    for (int q = 1; q <= (m == 2 ? 64 : 16); ++q) {
      if (kp && q != kp) continue;
      const int ktp = (KT + q - 1) / q, KP = (KT + ktp - 1) / ktp;
      if (!kp && KP > 1 && (KP != q || ktp < (m == 2 ? 3 : 4) || tiles * KP > 4 * (int64_t)cus)) continue;
      if (KP > 1 && !allow_split) continue;
      if (tiles * KP > 0x7fffffff / 256) continue;
      const size_t part = KP > 1 ? (size_t)KP * a.M * ld * 4 : 0;
      if (part > kMaxPartBytes) continue;
      const double t = estimate(a, m, tiles * KP, KP, ktp, 2.0 * (double)part / 1e6, cus);
      if (!best.ok || t < best.us) best = GemmnPlan{m, KP, ktp, part ? kCntBytesN + part : 0, t, true};
    }
  }
  return best;
}

hipError_t gemmn_launch(const LinearArgs& a, const GemmnPlan& pl, void* ws, hipStream_t s) {
  if (!pl.ok || (pl.KP > 1 && !ws)) return hipErrorInvalidValue;
  const int mb = pl.mb;
  const bool swi = a.epi == EPI_SWIGLU;
  GNArgs k{};
  k.A = (const _Float16*)a.A; k.lda = a.lda;
  k.W = (const unsigned char*)a.W; k.ldw = a.ldw;
  k.scales = (const _Float16*)a.scales; k.zeros = (const _Float16*)a.zeros;
  k.ep = a.epi_args();
  k.C = (_Float16*)a.C; k.ldc = a.ldc;
  k.M = a.M; k.N = a.N; k.K = a.K; k.G = a.G;
  k.F = swi ? a.N / 2 : a.N;
  k.gshift = a.G == 1 ? 31 : __builtin_ctz((unsigned)a.g);
  const int bm = 32 * mb, bno = swi ? GN_ROWS / 2 : GN_ROWS;
  k.nbm = (a.M + bm - 1) / bm;
  k.nbn = (k.F + bno - 1) / bno;
  k.gm = std::min(4, k.nbm);
  k.KT = (a.K + 63) / 64;
  const int64_t tiles = (int64_t)k.nbm * k.nbn;
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  k.KP = pl.KP; k.ktp = pl.ktp;
  k.part = pl.KP > 1 ? (float*)((char*)ws + kCntBytesN) : nullptr;
  k.up0 = (k.F + 7) & ~7;
  k.ldp = swi ? 2 * k.up0 : k.up0;
  const int nwg = (int)tiles * pl.KP;
  k.xcd = nwg % 8 == 0;
  k.vec_store = (a.ldc % 8 == 0) && (((uintptr_t)a.C & 15) == 0);
  k.vec_resid = (a.ldr % 8 == 0) && (((uintptr_t)a.resid & 15) == 0);
  const int64_t wrow = a.fmt == FMT_INT4 ? a.K / 2 : a.K;
  k.a_bytes = (uint32_t)(((int64_t)(a.M - 1) * a.lda + a.K) * 2);
  k.w_bytes = (uint32_t)((int64_t)(a.N - 1) * a.ldw + wrow);
  k.s_bytes = (uint32_t)((int64_t)a.N * a.G * 2);
  k.z_bytes = a.zeros ? k.s_bytes : 0u;
  if (a.fmt == FMT_INT4)
    return mb == 8 ? launch_mb<FMT_INT4, 8>(k, swi, nwg, s)
         : mb == 4 ? launch_mb<FMT_INT4, 4>(k, swi, nwg, s) : launch_mb<FMT_INT4, 2>(k, swi, nwg, s);
  return mb == 8 ? launch_mb<FMT_INT8, 8>(k, swi, nwg, s)
       : mb == 4 ? launch_mb<FMT_INT8, 4>(k, swi, nwg, s) : launch_mb<FMT_INT8, 2>(k, swi, nwg, s);
}

}  // namespace mq
