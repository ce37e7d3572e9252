// W4A16 MFMA GEMM in which every operand reaches the CU through a ring of LDS stages (fp16).
//
// One workgroup per CU owns 80 .. 128 rows of a block of 512 or 256 columns and walks K (or its share of
// K) in blocks of 128.  Everything a K block needs -- the activation rows, the packed
// weights, the group scales and zero-points -- is copied from global memory straight into a ring of LDS
// stages (global_load_lds, 16 B per lane, no staging registers) several K blocks ahead; the ring is the
// latency cover that a second workgroup per CU provides in the 64-row tile kernel.  Each of the eight
// wavefronts (two per SIMD: one wavefront alone issues an instruction every five or six clocks, too
// few for the matrix pipe) owns all row tiles of TW = 4 or 2 of the 16-column tiles: no weight is
// dequantised twice.  B operands are scaled, (q - z) * s rounded to fp16 -- the dequantised weight the
// operator is defined on -- so the matrix instructions accumulate in place.
//
// Used above 128 rows (MT = 5 .. 8 row tiles, TW = 2 or 4, workgroups of 256 or 512 columns) where a round model prices it below the
// 64-row tiles.  A K block of 8 x 4 tiles takes 3.0 us of which 1.1 do not depend on the rows (copies and dequantisation of the
// weights), so lower workgroups pay where they pad fewer rows or even out the rounds.  Every XCD takes a block of few rows and few
// columns of workgroups (tile_order): 2 % on average over 36 (layer, rows) points, 3 .. 8 % where the columns are not a multiple of
// eight workgroups (us, 128 x 256, dealt out in turn -> here: K 7168 x N 9344 at 600 / 743 rows 96.7 / 109.9 -> 88.8 / 102.1).  With TW = 4 an activation operand read from LDS feeds four matrix instructions instead of
// two -- the LDS reads per matrix instruction fall from 0.75 to 0.5 and the copies per column from a
// 128-row block of activations per 256 columns to one per 512 -- at the price of a ring of two stages
// instead of three and of registers: the 128 accumulators of the 8 x 4 tiles leave room for a ring of
// four activation operands and one set of packed weights, read twice per K block.
//
// The copies are issued from inline assembly, so the compiler does not know of them: it schedules and
// waits for the LDS reads itself (lgkmcnt), and the waits for the copies (vmcnt) are written by hand.
// No load that the compiler can see is in flight while a copy is (prologue and epilogue drain first).
#include "common.h"

#include <algorithm>

namespace mi355q {

int w4a16_splitk_reduce_launch(void* out, const float* partial, const void* bias, int M, int N, int splits,
                               int dtype, hipStream_t st);

namespace {

struct MidArgs {
  uint16_t* out;
  const uint16_t* x;
  const u4* qw;
  const uint16_t* scales;
  const void* zeros;
  const uint16_t* bias;
  int M, K, N;
  int kper;                   // K blocks per split
  TileOrder order;            // of the output tiles and splits
  uint32_t gpk, gpk_magic;    // K blocks per group and ceil(2^32 / gpk)
  float* partial;             // split K: fp32 tiles [split][M][N]; null: write the output
  int tall;                   // MIX kernels: the first workgroups' row tiles are one higher than the others'
  // IOBF kernels (bf16 rows staged as fp16 times a power of two each; scales, bias and output bf16):
  const float* row_scale;     // [M] the power of two each staged row has to be multiplied back by
  const uint32_t* scale_max;  // [64] largest scale magnitude (bf16 bits) of 64 slices of the scales array
};

// TW: 16-column tiles per wavefront -- 2: a workgroup of 256 columns; 4: of 512 columns.  MT: row tiles of 16 per workgroup
template <int TW, int MT>
struct MidCfg {
  static constexpr int BM = 16 * MT;
  static constexpr int XC = (MT + 1) / 2;             // activation copies (4 rows each) per wavefront and stage
  static constexpr int BNW = 128 * TW;                // columns per workgroup
  static constexpr int A_BYTES = XC * 8192;           // 128 halves per row (of an odd number of row tiles: and 16 rows that nobody reads)
  static constexpr int W_OFF = A_BYTES;               // 8 wavefronts x TW column tiles x 1 KiB
  static constexpr int SZ_OFF = A_BYTES + 8192 * TW;  // 8 wavefronts x (256 B of scales + 256 B of zero-points)
  static constexpr int STAGE = A_BYTES + 8192 * TW + 4096;
  static constexpr int D = (160 * 1024 - 1024) / STAGE < 6 ? (160 * 1024 - 1024) / STAGE : 6;   // stages in the ring
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

struct MidDq {
  uint32_t magic, mlo, mhi;
};

// Pair p (0..3) of one packed word -> two of the 8 weights of an MFMA K step, (q - z) * s in fp16,
// as the 32-bit word p of the B operand.  zlo = 1024 + z, zhi = 64 + z (PRESCALED: 1024 and 64, and
// zs = z * s is subtracted after the scaling).  Three or four instructions: the K loop deals them out
// between the matrix instructions instead of dequantising an operand in one burst.
template <int ZK>
__device__ __forceinline__ uint32_t mid_dequant_pair(uint32_t w, int p, _Float16 zlo1, _Float16 zhi1, _Float16 s1,
                                                     _Float16 zs1, const MidDq& k) {
  const h2 zlo = {zlo1, zlo1}, zhi = {zhi1, zhi1}, ss = {s1, s1}, zs = {zs1, zs1};
  const h2 sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const uint32_t ws = (p & 2) ? w >> 8 : w;
  h2 r;
  if (p & 1) {
    const h2 a = bitcast<h2>((ws & k.mhi) | k.magic);  // 1024 + 16 q
    r = __builtin_elementwise_fma(a, sixteenth, -zhi);
  } else {
    const h2 a = bitcast<h2>((ws & k.mlo) | k.magic);  // 1024 + q
    r = a - zlo;
  }
  if (ZK == MI355Q_ZP_PRESCALED) r = __builtin_elementwise_fma(r, ss, -zs);
  else r *= ss;
  return bitcast<uint32_t>(r);
}

// IOBF: the activations are bf16 rows that a pass before this kernel stored as fp16 times a power of
// two each; the scales are bf16 and become fp16 here, times one power of two for the whole array that
// brings the largest of them into [2^10, 2^11) -- (q - z) s stays below fp16's largest number and a
// scale 2^24 below the largest one still keeps all its bits; the epilogue undoes both powers of two
// exactly (one ldexp per output) and rounds to bf16.
template <int ZK, int TW, int MT, bool IOBF>
__device__ __forceinline__ void mid_tile(MidArgs a, const int m0, const int tn, const int split) {   // (by value: by reference the copies' addresses are made anew for every K block.  As the kernel itself
  // this was 4 .. 5 % slower with five and six row tiles of 512 columns, 4096 x 28672 at 333 rows 87.2 us, here 83.6)
  extern __shared__ __align__(16) unsigned char lds[];
  static_assert(!IOBF || ZK != MI355Q_ZP_PRESCALED, "pre-scaled zero-points stay with the bf16 kernel");
  typedef MidCfg<TW, MT> C;
  constexpr int D = C::D, STAGE = C::STAGE, XC = C::XC;
  constexpr bool HASZ = ZK != MI355Q_ZP_NONE;
  constexpr int NSLOT = XC + TW + 1;                  // copy slots per wavefront and stage (the last: scales + zeros)
  constexpr int NC = XC + TW + 1 + (HASZ ? 1 : 0);    // copy instructions per wavefront and stage
  static_assert((D - 1) * NC <= 63, "vmcnt is a 6-bit counter");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kq = lane >> 4;
  const int N = a.N, K = a.K, M = a.M, G = K >> 7;
  // N may end in the middle of a 256-column tile: the wavefronts of the missing slab work on the
  // previous one and their columns are never stored
  const int wslab = TW == 4 ? wave >> 1 : wave >> 2;                 // slab of the workgroup this wavefront works on
  const bool live = (tn * TW + wslab) < (N >> 7);
  const int slab = live ? tn * TW + wslab : (N >> 7) - 1;
  const int t0 = TW == 4 ? (wave & 1) * 4 : (wave & 3) * 2;          // first of this wavefront's TW tiles of the slab
  const int gb = split * a.kper, ge = min(G, gb + a.kper);
  const uint32_t lds_base =
      __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds);
  int sshift = 0;                                     // IOBF: scales are multiplied by 2^sshift
  if (IOBF) {
    uint32_t mx = a.scale_max[lane];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t other = (uint32_t)__shfl_xor((int)mx, o, 64);
      mx = mx > other ? mx : other;
    }
    const int expo = (int)(mx >> 7);
    if (mx != 0 && expo != 255) sshift = 10 - ((expo > 0 ? expo : 1) - 127);
    sshift = __builtin_amdgcn_readfirstlane(sshift);
  }

  // ---- copies.  Activations: one copy moves 4 rows of 256 B; lane = 16 * row + position, and position p
  // of row r receives the row's 16-byte chunk p ^ (r & 15), which keeps the MFMA operand reads (16 rows x
  // one chunk index per quarter wavefront) on 16 different bank groups.  Wavefront v copies row groups
  // v, v + 8, ...; rows past M re-read the last row (their results are never stored).
  uint32_t xo[XC];
#pragma unroll
  for (int p = 0; p < XC; ++p) {
    const int r = 4 * (wave + 8 * p) + (lane >> 4);
    const int row = min(m0 + r, M - 1);
    xo[p] = ((uint32_t)row * (uint32_t)K + 8u * (uint32_t)((lane & 15) ^ (r & 15))) * 2u;
  }
  const uint32_t lane16 = (uint32_t)lane * 16u;
  const uint32_t zlane = ZK == MI355Q_ZP_PACKED ? (uint32_t)(lane & 3) * 16u : lane16;
  const char* const xg = (const char*)a.x;
  const char* const wg = (const char*)a.qw + ((size_t)slab * G * 8 + t0) * 1024;
  const char* const sg = (const char*)a.scales + 256 * slab;
  const char* const zg = (const char*)a.zeros + (ZK == MI355Q_ZP_PACKED ? 64 : 256) * slab;
  const uint32_t zrow = ZK == MI355Q_ZP_PACKED ? (uint32_t)N / 2u : (uint32_t)N * 2u;
  // The workgroups of one split start together and stay roughly in step, and K block g of every
  // activation row lies a multiple of 8 KiB (Llama shapes) from that of the next: all of them would ask
  // the same few L2 channels for the same bytes at the same time.  Each column tile therefore walks its K
  // range from a different starting block (and wraps round): iteration i is K block gb + (rot + i) % nk.
  const int nk = ge - gb;
  const int rot = (int)((unsigned)tn % (unsigned)nk);
  auto copy_slot = [&](int s, int slot, int i) {
    const uint32_t sb = lds_base + (uint32_t)(slot * STAGE);
    int gq = rot + min(i, nk - 1);                    // past the end: a re-read into a stage nobody reads
    gq = gb + (gq >= nk ? gq - nk : gq);
    if (s < XC) {
      lds_copy16(xo[s < XC ? s : 0], xg + (size_t)gq * 256, sb + (uint32_t)((wave + 8 * s) * 1024));
    } else if (s < XC + TW) {
      const int t = s - XC;
      lds_copy16(lane16, wg + (size_t)gq * 8192 + t * 1024, sb + (uint32_t)(C::W_OFF + wave * 1024 * TW + t * 1024));
    } else {
      const uint32_t qrow = a.gpk_magic ? (uint32_t)(((uint64_t)(uint32_t)gq * a.gpk_magic) >> 32) : (uint32_t)gq;
      if (lane < 16) {
        lds_copy16(lane16, sg + (size_t)qrow * N * 2, sb + (uint32_t)(C::SZ_OFF + wave * 512));
        if (HASZ) lds_copy16(zlane, zg + (size_t)qrow * zrow, sb + (uint32_t)(C::SZ_OFF + wave * 512 + 256));
      }
    }
  };

  // ---- LDS reads (plain loads: the compiler places the waits)
  const uint32_t a_lane = (uint32_t)(c * 256);
  uint32_t a_pos[4];
#pragma unroll
  for (int st = 0; st < 4; ++st) a_pos[st] = a_lane + (uint32_t)(((4 * st + kq) ^ c) * 16);
  auto read_a = [&](int slot, int mt, int st) {
    return bitcast<h8>(*(const u4*)(lds + slot * STAGE + a_pos[st] + mt * 4096));
  };
  auto read_w = [&](u4 (&w)[TW], int slot) {
#pragma unroll
    for (int t = 0; t < TW; ++t) w[t] = *(const u4*)(lds + slot * STAGE + C::W_OFF + wave * 1024 * TW + t * 1024 + lane * 16);
  };
  struct Sz { uint2 s; uint2 zs; uint32_t z; };
  auto read_sz = [&](Sz& q, int slot) {
    const unsigned char* p = lds + slot * STAGE + C::SZ_OFF + wave * 512;
    if (TW == 4) q.s = *(const uint2*)(p + (8 * c + t0) * 2);
    else q.s.x = *(const uint32_t*)(p + (8 * c + t0) * 2);
    if (ZK == MI355Q_ZP_PACKED) q.z = *(const uint32_t*)(p + 256 + c * 4) >> (4 * t0);
    if (ZK == MI355Q_ZP_PRESCALED) {
      if (TW == 4) q.zs = *(const uint2*)(p + 256 + (8 * c + t0) * 2);
      else q.zs.x = *(const uint32_t*)(p + 256 + (8 * c + t0) * 2);
    }
  };
  // per column tile: scale, 1024 + z, 64 + z, z * s
  _Float16 sc[TW], zlo[TW], zhi[TW], zsc[TW];
  auto prep = [&](const Sz& q) {
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const uint32_t sw = t < 2 ? q.s.x : q.s.y;
      if (IOBF) sc[t] = (_Float16)__builtin_ldexpf(bitcast<float>((t & 1) ? (sw & 0xffff0000u) : (sw << 16)), sshift);
      else sc[t] = bitcast<_Float16>((uint16_t)((t & 1) ? (sw >> 16) : (sw & 0xffffu)));
      if (ZK == MI355Q_ZP_PRESCALED) {
        const uint32_t zw = t < 2 ? q.zs.x : q.zs.y;
        zsc[t] = bitcast<_Float16>((uint16_t)((t & 1) ? (zw >> 16) : (zw & 0xffffu)));
        zlo[t] = (_Float16)1024.0f;
        zhi[t] = (_Float16)64.0f;
      } else {
        // fp16 bit patterns directly: 1024 + z = 0x6400 | z, 64 + z = 0x5400 | z << 4
        const uint32_t z = ZK == MI355Q_ZP_PACKED ? (q.z >> (4 * t)) & 15u : 8u;
        zlo[t] = bitcast<_Float16>((uint16_t)(0x6400u | z));
        zhi[t] = bitcast<_Float16>((uint16_t)(0x5400u | (z << 4)));
        zsc[t] = (_Float16)0.0f;
      }
    }
  };
  MidDq dqk = {0x64006400u, 0x000f000fu, 0x00f000f0u};
  asm volatile("" : "+v"(dqk.magic));
  asm volatile("" : "+s"(dqk.mlo));
  asm volatile("" : "+s"(dqk.mhi));

  f4 acc[MT][TW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < TW; ++t) acc[mt][t] = (f4){0.f, 0.f, 0.f, 0.f};

  // ---- prologue: the whole ring is requested, the first stage awaited
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int s = 0; s < NSLOT; ++s) copy_slot(s, d, d);
  wait_vmcnt<(D - 1) * NC>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // A operands travel through a small ring of registers: group j (K step j / MT, row tile j % MT) uses
  // entry j % R and requests the operand of group j + PF.  A whole K step ahead where the registers
  // allow (R = 2 MT entries); with four column tiles per wavefront the 128 accumulator registers leave
  // room for a ring of four, three groups (twelve matrix instructions) ahead -- and for one set of
  // packed weights instead of two, re-read when its last word has been dequantised.
  constexpr int PF = TW == 4 ? 3 : MT, R = TW == 4 ? 4 : 2 * MT;
  constexpr bool WDB = TW != 4;                        // two sets of packed weights that swap roles per K block
  static_assert((4 * MT) % R == 0, "the ring index of a group is the same in every K block");
  u4 w0[TW], w1[WDB ? TW : 1];
  Sz sz;
  h8 av[R];
  u4 bv[2][TW];
  read_w(w0, 0);
  read_sz(sz, 0);
#pragma unroll
  for (int j = 0; j < PF; ++j) av[j % R] = read_a(0, j % MT, j / MT);
  prep(sz);
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int p = 0; p < 4; ++p) bv[0][t][p] = mid_dequant_pair<ZK>(w0[t][0], p, zlo[t], zhi[t], sc[t], zsc[t], dqk);

  constexpr int NP = 4 * TW;                          // operand words dequantised per K step, dealt out over the MT groups
  constexpr int JX = 4 * MT - PF;                     // first group whose request goes to the next stage
  constexpr int CPG = (NSLOT + PF - 1) / PF;          // copy slots issued per group from there on
  int slot = 0;
  // One K block: four K steps of MT groups of TW matrix instructions, with the group's other work dealt
  // out behind them (a matrix instruction occupies its pipe for four issue slots).  While step st
  // multiplies, the B operands of step st + 1 are dequantised.  In step 2 the wavefront's own copies of
  // the next stage are awaited and its scales (and, with two weight sets, packed weights) read.  Before
  // group JX every LDS read of this stage has been issued and awaited: after the barrier there the stage
  // is refilled with K block i + D while the first A operands of block i + 1 are requested.
  auto kblock = [&](int i, u4 (&wc)[TW], u4 (&wn)[TW]) __attribute__((always_inline)) {
    const int nslot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int cur = st & 1, nxt = cur ^ 1;
      if (st == 2) {
        wait_vmcnt<(D - 2) * NC>();
        if (WDB) read_w(wn, nslot);
        read_sz(sz, nslot);
      }
      if (st == 3) {
        if (!WDB) read_w(wn, nslot);                  // (its own copies: no barrier needed; wc and wn are one array)
        prep(sz);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int j = st * MT + mt, jn = j + PF;
        if (j == JX) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[j % R], bitcast<h8>(bv[cur][t]), acc[mt][t], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (t == 0) {
            av[jn % R] = jn < 4 * MT ? read_a(slot, jn % MT, jn / MT) : read_a(nslot, (jn - 4 * MT) % MT, (jn - 4 * MT) / MT);
            if (j >= JX) {
#pragma unroll
              for (int sl = (j - JX) * CPG; sl < (j - JX + 1) * CPG && sl < NSLOT; ++sl) copy_slot(sl, slot, i + D);
            }
          }
          // the operand words of this group (word q belongs to group q * MT / NP), dealt out over its TW slices
          int k = 0;
#pragma unroll
          for (int q = 0; q < NP; ++q) {
            if (q * MT / NP != mt) continue;
            if (k++ % TW != (t + 1) % TW) continue;
            const int tt = q >> 2, p = q & 3;
            bv[nxt][tt][p] = mid_dequant_pair<ZK>(st < 3 ? wc[tt][st + 1] : wn[tt][0], p, zlo[tt], zhi[tt], sc[tt], zsc[tt], dqk);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    slot = nslot;
  };
  for (int i = 0;; i += 2) {
    if (WDB) kblock(i, w0, (u4(&)[TW])w1);
    else kblock(i, w0, w0);
    if (i + 1 >= nk) break;
    if (WDB) kblock(i + 1, (u4(&)[TW])w1, w0);
    else kblock(i + 1, w0, w0);
    if (i + 2 >= nk) break;
  }
  // no copy may still be writing LDS when the workgroup retires, and none may be in flight next to the
  // loads below
  wait_vmcnt<0>();

  // ---- epilogue through LDS (the ring is free now): a lane holds TW adjacent columns of 4 rows per row
  // tile, which as stores would touch a few bytes in every 32; written to an fp32 tile in LDS and read
  // back row by row, every store instruction writes whole rows of the workgroup's columns.  (512 columns:
  // the tile goes through in two halves of 64 rows.)
  constexpr int EP = C::BNW * 4 + 16;                  // bytes per tile row in LDS
  constexpr int HALVES = TW == 4 ? 2 : 1, MTH = (MT + HALVES - 1) / HALVES;
  static_assert(16 * MTH * EP <= D * STAGE, "the output tile fits in the ring");
  constexpr int IPR = C::BNW / 256;                    // instructions per row, 4 columns per lane
  typedef Elem<IOBF ? MI355Q_BF16 : MI355Q_F16> IO;
  f4 bs[IPR];
#pragma unroll
  for (int q = 0; q < IPR; ++q) {
    bs[q] = (f4){0.f, 0.f, 0.f, 0.f};
    const int col = tn * C::BNW + 4 * lane + 256 * q;
    if (a.bias && !a.partial && col < N) {
      const uint2 bw = *(const uint2*)(a.bias + col);
      bs[q] = (f4){IO::to_f32((uint16_t)(bw.x & 0xffffu)), IO::to_f32((uint16_t)(bw.x >> 16)),
                   IO::to_f32((uint16_t)(bw.y & 0xffffu)), IO::to_f32((uint16_t)(bw.y >> 16))};
    }
  }
#pragma unroll
  for (int h = 0; h < HALVES; ++h) {
    __syncthreads();                                   // every wavefront has left the K loop (or the half before)
    {
      unsigned char* base = lds + (128 * wslab + 8 * c + t0) * 4;
#pragma unroll
      for (int mh = 0; mh < MTH; ++mh)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mt = h * MTH + mh;
          if (mt >= MT) continue;
          unsigned char* q = base + (mh * 16 + 4 * kq + i) * EP;
          if (TW == 4) *(f4*)q = (f4){acc[mt][0][i], acc[mt][1][i], acc[mt][2 % TW][i], acc[mt][3 % TW][i]};
          else *(f2*)q = (f2){acc[mt][0][i], acc[mt][1][i]};
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2 * MTH; ++p) {
      const int r = wave + 8 * p, m = m0 + h * 16 * MTH + r;
      if (m >= min(M, m0 + C::BM)) break;
      // IOBF: the row's power of two and the scales' in one exponent
      int back = 0;
      if (IOBF) back = (int)((bitcast<uint32_t>(a.row_scale[m]) >> 23) & 255u) - 127 - sshift;
#pragma unroll
      for (int q = 0; q < IPR; ++q) {
        const int col = tn * C::BNW + 4 * lane + 256 * q;
        if (col >= N) continue;
        f4 v = *(const f4*)(lds + r * EP + lane * 16 + 1024 * q);
        if (IOBF) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = __builtin_ldexpf(v[e], back);
        }
        if (a.partial) {
          *(f4*)(a.partial + ((size_t)split * M + m) * N + col) = v;
        } else {
          uint2 o;
          o.x = (uint32_t)IO::from_f32(v[0] + bs[q][0]) | ((uint32_t)IO::from_f32(v[1] + bs[q][1]) << 16);
          o.y = (uint32_t)IO::from_f32(v[2] + bs[q][2]) | ((uint32_t)IO::from_f32(v[3] + bs[q][3]) << 16);
          *(uint2*)(a.out + (size_t)m * N + col) = o;
        }
      }
    }
  }
}

// MIX: workgroups of MT row tiles for the first rows and of MT - 1 for the others
template <int ZK, int TW, int MT, bool IOBF, bool MIX>
__global__ void __launch_bounds__(512, 1)
w4a16_mid_kernel(MidArgs a) {
  int tm, tn, split;
  a.order.locate(blockIdx.x, tm, tn, split);
  if constexpr (MIX) {
    if (tm >= a.tall) {
      mid_tile<ZK, TW, MT - 1, IOBF>(a, 16 * (a.tall + tm * (MT - 1)), tn, split);
      return;
    }
  }
  mid_tile<ZK, TW, MT, IOBF>(a, 16 * MT * tm, tn, split);
}

template <int ZK, int TW, int MT, bool IOBF, bool MIX>
int launch_mid(MidArgs a, int mtiles, int splits, hipStream_t st) {
  typedef MidCfg<TW, MT> C;
  typedef MidCfg<TW, MIX ? MT - 1 : MT> L;
  const size_t shmem = std::max((size_t)C::D * C::STAGE, (size_t)L::D * L::STAGE);
  static hipError_t attr = hipFuncSetAttribute((const void*)w4a16_mid_kernel<ZK, TW, MT, IOBF, MIX>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  MQ_REQUIRE(attr == hipSuccess, "w4a16_gemm(mid): cannot reserve %zu bytes of LDS: %s", shmem, hipGetErrorString(attr));
  const int ntiles = (a.N + C::BNW - 1) / C::BNW;
  a.order = tile_order(mtiles, ntiles, splits, (double)C::BM * a.kper * 256, (double)C::BNW * a.kper * 64);
  hipLaunchKernelGGL((w4a16_mid_kernel<ZK, TW, MT, IOBF, MIX>), dim3((unsigned)(mtiles * ntiles * splits)), dim3(512), shmem, st, a);
  MQ_LAUNCH_CHECK("w4a16_gemm(mid)");
  return 0;
}
template <int ZK, int TW, int MT, bool IOBF>
int launch_mid_rows(MidArgs a, int mixed, int splits, hipStream_t st) {
  if constexpr (TW == 4 && MT == 8)
    if (mixed) {
      a.tall = (a.M + 15) / 16 - mixed * (MT - 1);
      return launch_mid<ZK, TW, MT, IOBF, true>(a, mixed, splits, st);
    }
  return launch_mid<ZK, TW, MT, IOBF, false>(a, (a.M + 16 * MT - 1) / (16 * MT), splits, st);
}

// mt: row tiles of a workgroup; from bit 8 on the workgroups per column tile, where some of them take one row tile less (0: none does).  Of 512 columns and
// eight row tiles, where layers of several rounds go.
bool mid_mixes(int M, int tw, int mt, int mixed) {
  const int S = (M + 15) / 16;
  return tw == 4 && mt == 8 && mixed * (mt - 1) < S && S < mixed * mt;
}
template <int ZK, bool IOBF>
int launch_mid_tw(const MidArgs& a, int tw, int mt, int splits, hipStream_t st) {
  const int mixed = mid_mixes(a.M, tw, mt & 255, mt >> 8) ? mt >> 8 : 0;
#define MQ_MID(MT) case MT: return tw == 4 ? launch_mid_rows<ZK, 4, MT, IOBF>(a, mixed, splits, st) : launch_mid_rows<ZK, 2, MT, IOBF>(a, mixed, splits, st)
  switch (mt & 255) {
    MQ_MID(5);
    MQ_MID(6);
    MQ_MID(7);
    default:
    MQ_MID(8);
  }
#undef MQ_MID
}

}  // namespace

// Row tiles of 16 and column tiles of 16 per wavefront of a workgroup, and K splits: the cheapest by a price in us, with the partial
// tiles within `bytes`.  A round of workgroups (one per CU) pays a step per K block -- weights and their dequantisation, and a part
// that grows with the rows --, the last one by the share of the chip that it occupies; a split pays for its second launch and the bytes of its
// partial tiles, and a chip that stays full runs at a lower clock.  Lower workgroups than 128 rows pad fewer rows and make more even rounds.  Measured (us, 128 rows -> here, packed zero-points,
// groups of 128): K 4096 x N 28672 at 170 / 333 / 800 rows 54.8 / 95.9 / 202.9 -> 47.0 / 87.2 / 183.9; K 3584 x N 37888 at 333 / 1000
// 97.3 / 274.4 -> 90.2 / 264.6; K 18944 x N 3584 at 333 / 1000 60.4 / 149.3 -> 58.3 / 139.9; K 8192 x N 10240 at 333 / 512 68.8 / 101.6 ->
// 65.7 / 99.6; four column tiles with a split, K 28672 x N 8192 at 1400: 623 -> 591 (six row tiles, six ranges).
// Fitted to 5844 launches (12 layers, 130 .. 2048 rows, 5 .. 8 row tiles, 1 .. 6 splits), rms error 3 %; the pick is within 0.4 % of the
// best of them on average, and 6 % faster than the best one of 128 rows.
struct MidPlan {
  int tw, mt, splits;
  double price;
};
struct MidPrice {
  double full, full_mt, lone, lone_mt, odd, base, round, power, split, split_mn;
};
static constexpr MidPrice kMid[2] = {{0.391, 0.1518, 0.498, 0.1003, 0.047, 4.89, 2.44, 0.00330, 2.10, 0.98},
                                     {1.041, 0.2372, 1.211, 0.1730, -0.034, 7.09, 2.40, 0.00409, 1.05, 0.92}};
constexpr double kMixed = 1.02;      // what their price has to be below the others' by
static MidPlan make_mid_plan(int M, int K, int N, size_t bytes) {
  const int G = K / 128, cus = device_cu_count(), S = (M + 15) / 16;
  MidPlan best = {2, 8, 1, 1e30};
  double least = 1e30;
  // rows: workgroups per column tile, `mean` row tiles high; mixed: some of mt and some of mt - 1
  auto offer = [&](int tw, int mt, int rows, double mean, bool mixed) {
    const int tiles = rows * ((N + 128 * tw - 1) / (128 * tw));
    const MidPrice& p = kMid[tw == 4];
    const double odd = p.odd * (mixed ? 0.5 : mt & 1), full = p.full + p.full_mt * mean + odd, lone = p.lone + p.lone_mt * mean + odd;
    for (int s = 1; s <= 8 && (s == 1 || ((long)tiles * (s - 1) < 6L * cus && G / s >= 4 && (size_t)s * M * N * sizeof(float) <= bytes)); ++s) {
      const int kper = (G + s - 1) / s;
      if (s > 1 && (s - 1) * kper >= G) continue;    // an empty split
      const int wgs = tiles * s, rounds = wgs / cus;
      const double rest = (double)(wgs - rounds * cus) / cus;
      double t = kper * (rounds * full + (rest > 0 ? lone + (full - lone) * rest * rest : 0.0)) * (1 + p.power * mean * std::min(rounds, 6)) +
                 p.round * (rounds + (rest > 0)) + p.base;
      if (s > 1) t += p.split + p.split_mn * 1e-6 * s * M * N;
      if (mixed) t = kMixed * t + kper * p.full_mt * (mt - mean);     // (a CU with one high workgroup more than the others)
      if (t < least) {
        least = t;
        best = {tw, mixed ? mt | rows << 8 : mt, s, mixed ? best.price : t};
      }
    }
  };
  for (int tw = 2; tw <= 4; tw += 2)
    for (int mt = 5; mt <= 8; ++mt) offer(tw, mt, (M + 16 * mt - 1) / (16 * mt), mt, false);
  // (the price stays that of the even ones: other kernels are chosen by it, whose operands are exact, and what is rounded to fp16 shall not
  // depend on how the rows are dealt out)
  // Even rounds by workgroups of 7 and 8 row tiles, up to three rounds: a chip that is full for longer runs into its power limit and gains nothing.  (us, all of 128
  // rows -> here: 3584 x 37888 at 700 rows 191.4 -> 187.2, 4096 x 28672 at 1024 / 1537, bf16, 228.6 / 337.4 -> 224.8 / 336.3, 8192 x 28672 at 1024 435.1 -> 419.2; in four rounds
  // 4096 x 28672 at 2048 437.3 / 437.9.  Of 256 columns, and 6 and 7 or 5 and 6 row tiles: within 1 % on average.)
  for (int rows = S / 8 + 1; rows <= 127 && mid_mixes(M, 4, 8, rows) && (long)rows * ((N + 511) / 512) <= 3L * cus; ++rows) offer(4, 8, rows, (double)S / rows, true);
  return best;
}
// (bytes: 0, what a fixed scratch of 32 MiB leaves, or 64 MiB, but for callers with less than the library asked for)
MidPlan w4a16_mid_plan(int M, int K, int N, size_t bytes) {
  const int mib = (int)(bytes >> 20);
  if (bytes & 0xfffff || (mib != 0 && mib != 31 && mib != 64)) return make_mid_plan(M, K, N, bytes);
  return cached_plan(mib, M, N, K, [](int mib, int M, int N, int K) { return make_mid_plan(M, K, N, (size_t)mib << 20); });
}

// fp16 activations, group sizes that are multiples of 128.  `splits` 0: as many as fit the chip in one
// round (one workgroup per CU), each at least four K blocks long and the partial tiles within 64 MiB.
int w4a16_mid_launch(void* out, const void* x, const int32_t* qweight, const void* scales, const void* zeros,
                     int zeros_kind, const void* bias, int M, int K, int N, int group_size, int dtype,
                     void* workspace, size_t workspace_bytes, int splits, int tw, int mt, hipStream_t st) {
  MQ_REQUIRE(dtype == MI355Q_F16 && group_size % 128 == 0,
             "w4a16_gemm(mid): fp16 and group sizes that are multiples of 128 only (dtype %d, group %d)", dtype, group_size);
  MQ_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32), "w4a16_gemm: activation matrix %d x %d is 4 GiB or more", M, K);
  const int G = K / 128;
  if (tw != 4) tw = 2;
  if ((mt & 255) < 5 || (mt & 255) > 8) mt = 8;
  if (splits <= 0) {
    const long wgs = (long)((M + 16 * (mt & 255) - 1) / (16 * (mt & 255))) * ((N + 128 * tw - 1) / (128 * tw));
    splits = (int)std::min<long>(device_cu_count() / wgs, G / 4);
    while (splits > 1 && (size_t)splits * M * N * sizeof(float) > ((size_t)64 << 20)) --splits;
    if (splits < 1) splits = 1;
  }
  if (splits > G) splits = G;
  if (splits > 1 && (!workspace || workspace_bytes < (size_t)splits * M * N * sizeof(float))) splits = 1;
  MidArgs a = {};
  a.out = (uint16_t*)out;
  a.x = (const uint16_t*)x;
  a.qw = (const u4*)qweight;
  a.scales = (const uint16_t*)scales;
  a.zeros = zeros;
  a.bias = (const uint16_t*)bias;
  a.M = M; a.K = K; a.N = N;
  a.kper = (G + splits - 1) / splits;
  splits = (G + a.kper - 1) / a.kper;                  // no empty splits
  a.gpk = (uint32_t)group_size / 128u;
  a.gpk_magic = a.gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + a.gpk - 1) / a.gpk) : 0u;
  a.partial = splits > 1 ? (float*)workspace : nullptr;
  int rc;
  if (zeros_kind == MI355Q_ZP_NONE) rc = launch_mid_tw<MI355Q_ZP_NONE, false>(a, tw, mt, splits, st);
  else if (zeros_kind == MI355Q_ZP_PACKED) rc = launch_mid_tw<MI355Q_ZP_PACKED, false>(a, tw, mt, splits, st);
  else rc = launch_mid_tw<MI355Q_ZP_PRESCALED, false>(a, tw, mt, splits, st);
  if (rc) return rc;
  if (splits > 1) return w4a16_splitk_reduce_launch(out, (const float*)workspace, bias, M, N, splits, dtype, st);
  return 0;
}

// The same kernels on bf16 rows that the caller staged as fp16 (x16, one power of two per row in
// row_scale); scales, bias and output are bf16, scale_max holds the largest scale magnitude of 64 slices
// of the scales array.  Workgroups of 16 mt rows and 256 (tw 2) or 512 (tw 4) columns, K unsplit.
int w4a16_mid_launch_staged(void* out, const void* x16, const int32_t* qweight, const void* scales, const void* zeros,
                            int zeros_kind, const void* bias, int M, int K, int N, int group_size,
                            const float* row_scale, const uint32_t* scale_max, int tw, int mt, hipStream_t st) {
  MQ_REQUIRE(group_size % 128 == 0 && zeros_kind != MI355Q_ZP_PRESCALED && row_scale && scale_max && M > 64,
             "w4a16_gemm(mid, bf16 staged): group %d, zero-point kind %d, M %d not covered", group_size, zeros_kind, M);
  MidArgs a = {};
  a.out = (uint16_t*)out;
  a.x = (const uint16_t*)x16;
  a.qw = (const u4*)qweight;
  a.scales = (const uint16_t*)scales;
  a.zeros = zeros;
  a.bias = (const uint16_t*)bias;
  a.M = M; a.K = K; a.N = N;
  a.kper = K / 128;
  a.gpk = (uint32_t)group_size / 128u;
  a.gpk_magic = a.gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + a.gpk - 1) / a.gpk) : 0u;
  a.row_scale = row_scale;
  a.scale_max = scale_max;
  return zeros_kind == MI355Q_ZP_NONE ? launch_mid_tw<MI355Q_ZP_NONE, true>(a, tw, mt, 1, st)
                                      : launch_mid_tw<MI355Q_ZP_PACKED, true>(a, tw, mt, 1, st);
}

}  // namespace mi355q
