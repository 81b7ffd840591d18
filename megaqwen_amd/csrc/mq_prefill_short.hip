// Short prompts (up to SHORT_MAX_S tokens): every layer of the prefill in one launch.
//
// A layer of a short prompt is five dependent steps of a few microseconds each. As launches of
// their own they cost what a launch costs: the boundary (3.6 us between dependent launches of 256
// workgroups that load and store one word a lane), the first weight tile's trip from HBM, the
// drain; 40-50 us a layer against 4.5 us for reading its weights. Here the steps are tasks of
// one launch, on blocks of 16 prompt rows:
//   qkv   one head: input RMSNorm, product, QK-norm and RoPE, K/V append
//   attn  16 query rows of one head over all their keys
//   o     64 columns of o_proj, residual add
//   gu    64 MLP units: post-attention RMSNorm, gate and up products, SiLU(gate) * up
//   down  32 columns of down_proj, residual add
// A task of a product loads its weight rows into registers first (the whole k range: 8 waves x
// up to 128 registers), then waits for the tasks it reads from, loads the activation rows into
// LDS and multiplies. So the weights come from HBM while earlier tasks run (each XCD's list of tasks
// is 31 workgroups ahead), and a step costs a hand-over between workgroups instead of a launch.
// Whole prefill, same box, before (mq_prefill.hip's launches) -> now, us:
//   S = 1 1137 -> 626, 23 1285 -> 713, 64 1359 -> 773, 128 1451 -> 966, 200 1536 -> 1200, 256 1620 -> 1391
// (the launches win from about 330 tokens: a task's weights serve 16 rows at a time here).
// What bounds it: the chain of a layer's steps (S = 23: 22.5 us, of which about 7 us are the
// five hand-overs, 1.1 us twice the RMSNorm's VALU work, 0.9 us twice the LDS reads of a product's
// 16 rows by eight waves, the rest the activation rows' loads, the epilogues and the
// attention's chain); from 128 tokens also the 31 workgroups an XCD has for its tasks.
//
// Order and progress. XCD g owns KV group g and an eighth of the columns of every product, so
// the tasks that share weight rows share an L2. Each XCD's tasks form one list, ordered by
// layer and step; a workgroup takes the next task of its XCD's list with an atomic ticket and
// finishes it before it takes another. A task waits only for tasks of earlier steps, so the
// earliest unfinished task is either running or next on its XCD's list. A workgroup keeps its CU
// until its list is done (128 KB of LDS: one a CU), so this makes progress if every XCD has a
// workgroup for its list and one for its relay, and only then: where launches overlap, two of them
// could each hold a whole XCD that the other needs. So no task publishes anything before the
// launch has seen two of its workgroups on every XCD; they stay to the end. Where it has not seen
// them after PLACE_TICKS (other launches hold the CUs, or the device shows fewer XCDs), it runs
// from a single list instead (run_tasks<true>): all XCDs' tasks in the same order, each taken by
// whatever workgroup comes next, and every hand-over device-wide. The earliest unfinished task is
// then running or next for any workgroup, so one resident workgroup is enough. Polls are bounded
// all the same.
//
// Hand-over. Activations that cross XCDs are written with device-scope (sc1) stores and read
// with sc1 loads (no stale word in 2e8 reads, and as fast as L2 reads when many CUs read the
// same rows: 112 GB/s a CU either way; invalidating the L2 instead costs 15 us); q, K and V stay in
// their XCD (from a single list they cross XCDs too, and are written and read likewise). A task's stores are complete (vmcnt(0)) before its flag, layer + 1, is stored. The
// buffers are rewritten every layer; a task that overwrites rows depends, through the flags of
// those rows, on every task that read them (h: o and down of a row block follow all qkv,
// respectively gu, tasks of it; q, attention rows and MLP rows likewise).
//
// Numerics: every product is the same MFMA chain over k as in mq_prefill.hip (o_proj and
// down_proj: four quarter chains added in order), the norms, rotations, softmax and roundings
// the same operations in the same order, so a row's results are the same bits whatever path
// its prompt takes.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "megaqwen_amd.h"
#include "mq_common.h"
#include "mq_prefill_short.h"

namespace mq {
namespace ps {

constexpr int NW = 8, NT = 64 * NW, NXCD = 8, NWG = 256;
constexpr int RING = 8, STAGE = 2048;  // weight staging: stages in flight a wave, bytes of one (16 rows x 64 k)
constexpr int LDS_BYTES = NW * RING * STAGE;
// A column slice's row blocks are dealt to at most this many tasks, each of which loads the
// slice's weights: 4 x (4 + 2 + 6 + 4) tasks of the products a layer and XCD
constexpr int GROUPS = 4;
constexpr uint32_t POLL_LIMIT = 1u << 21;  // about 1 s of polling
// How long a launch waits for two workgroups on every XCD (100 MHz ticks: 100 us; on an idle
// device they are there within a few microseconds)
constexpr uint64_t PLACE_TICKS = 10000;

// Words of `sync` (device scope): per XCD a cache line with its ticket and role counters; the
// dead word, the launch's mode and the single list's ticket; then, for each step and relay wave, a
// line with one word per XCD.
enum : int { S_ATT = 0, S_O = 1, S_GU = 2, S_DOWN = 3, NSTEP = 4 };
constexpr int SY_ROLE = 1, SY_DEAD = DEAD_WORD, SY_MODE = 32 + 16, SY_ANY = 64 + 16, SY_STEPS = 32 * NXCD, SY_LINE = 16;
constexpr int SYNC_WORDS = SY_STEPS + NSTEP * NW * SY_LINE;
enum : uint32_t { MODE_XCD = 1, MODE_ANY = 2 };  // a list per XCD; a single list
static_assert(SYNC_WORDS <= H, "the sync area fits one row of fp32 partial sums");
// Words of `local`, one region per XCD that only its own workgroups touch: per step and relay
// wave the relay's word, then the flags of the XCD's tasks, per row block.
constexpr int NQKV = 4, NATT = 2, NO = 2, NGU = 6, ND = 4;  // an XCD's tasks of a step
__host__ __device__ constexpr int pad32(int n) { return (n + 31) / 32 * 32; }
__host__ __device__ constexpr int local_words(int nb) { return pad32(NSTEP * NW) + pad32((NQKV + NATT + NO + NGU + ND) * nb); }
static_assert(NXCD * local_words(1) <= H / 2, "the local area fits one row of bf16 activations");

struct Sync {
  int steps;                       // this XCD's word of the first line in `sync`
  int relay;                       // this XCD's relay words in `local` (NW a step)
  int qkv, att, o, gu, down;       // and its flags of each step
  __device__ Sync(int nb, int g) {
    steps = SY_STEPS + g;
    relay = g * local_words(nb);
    qkv = relay + pad32(NSTEP * NW);
    att = qkv + nb * NQKV;
    o = att + nb * NATT;
    gu = o + nb * NO;
    down = gu + nb * NGU;
  }
};

// One 16-byte LDS DMA per lane (see dma16) from a wave-uniform base plus the lane's byte offset:
// the base stays in scalar registers, which the weights in flight leave free. sc1: device scope.
__device__ __forceinline__ void dma16_at(const uint16_t* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(base), "s"(lds)
      : "memory");
}
__device__ __forceinline__ void dma16_at_sc1(const uint16_t* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2 sc1\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(base), "s"(lds)
      : "memory");
}
__device__ __forceinline__ void dma16_at_nt(const uint16_t* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(base), "s"(lds)
      : "memory");
}
// data of this XCD's own workgroups: past the CU's L1, served by the XCD's L2; or (ANY) of any XCD's
template <bool ANY>
__device__ __forceinline__ u32x4 ld4_xcd(const Buf& b, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(b.r, off, 0, ANY ? SC1 : 2 /* nt */);
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ u32x4 lds16(const uint8_t* p) { return *reinterpret_cast<const u32x4*>(p); }

// The lane's MFMA operands of a tile of rows in LDS (row r's 16-byte chunk c in slot
// c ^ (r % 8) of each 128 bytes): row r16 of a 16-row block, chunk 8 s + 4 ks + kg (k
// step ks of stage s) from operand pointer ks, 128 bytes a stage
struct Operand {
  const uint8_t* p[2];
  __device__ __forceinline__ Operand(const uint8_t* tile, int pitch, int r16, int kg) {
#pragma unroll
    for (int ks = 0; ks < 2; ks++) p[ks] = tile + r16 * pitch + 16 * ((4 * ks + kg) ^ (r16 & 7));
  }
  __device__ __forceinline__ u32x4 at(int ks, int bytes) const { return lds16(p[ks] + bytes); }
};

// NS stages of weight rows into registers as MFMA operands: stage i is 16 rows (pitch `pitch`
// elements, from p) by the 64 k from element off(i). Each goes through a 2 KB slot of the wave's
// own ring (two 1 KB DMAs of whole 128-byte row pieces; 16-byte chunk c of row r in slot
// c ^ (r % 8), so a fragment read is free of bank conflicts), RING stages in flight.
template <int NS, class Off>
__device__ __forceinline__ void load_weights(u32x4 (&b)[NS][2], const uint16_t* p, int pitch, Off off, uint8_t* ring,
                                             int lane) {
  const int r8 = lane >> 3, r16 = lane & 15, kg = lane >> 4;
  p = uniform_ptr(p);
  const uint32_t o0 = 2u * (uint32_t)(r8 * pitch + 8 * ((lane & 7) ^ r8));
  const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  const Operand w(ring, 128, r16, kg);
  auto issue = [&](int i) {
    const uint16_t* s = p + off(i);
    dma16_at(s, o0, l0 + STAGE * (i % RING));
    dma16_at(s + (size_t)8 * pitch, o0, l0 + STAGE * (i % RING) + 1024);
  };
#pragma unroll
  for (int i = 0; i < (NS < RING ? NS : RING); i++) issue(i);
#pragma unroll
  for (int i = 0; i < NS; i++) {
    // stages up to min(NS, i + RING) have been issued, two DMAs each
    switch (2 * ((NS < i + RING ? NS : i + RING) - i - 1)) {
      case 14: wait_vm<14>(); break;
      case 12: wait_vm<12>(); break;
      case 10: wait_vm<10>(); break;
      case 8: wait_vm<8>(); break;
      case 6: wait_vm<6>(); break;
      case 4: wait_vm<4>(); break;
      case 2: wait_vm<2>(); break;
      default: wait_vm<0>(); break;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ks++) b[i][ks] = w.at(ks, STAGE * (i % RING));
    if (i + RING < NS) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
      issue(i + RING);
    }
  }
}

// ROWS activation rows of K elements (rows past the prompt repeat its last one) into LDS, row r
// at r * 2 K bytes, its 16-byte chunk c in slot c ^ (r % 8). Returns with this wave's rows landed.
template <int K, int ROWS>
__device__ __forceinline__ void load_rows(const uint16_t* a, int row0, int S, uint8_t* lds, int wv, int lane) {
  constexpr int PPR = K / 512, N = ROWS * PPR / NW;  // 1 KB pieces a row, DMAs a wave
  const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
#pragma unroll
  for (int n = 0; n < N; n++) {
    const int i = wv + NW * n, r = i / PPR, part = i % PPR;
    dma16_at_sc1(a + (size_t)min(row0 + r, S - 1) * K + 512 * part, 16u * (uint32_t)(lane ^ (r & 7)), l0 + 1024u * (uint32_t)i);
  }
  wait_vm<0>();
}

// acc[c] += the products of the tile's 16 rows and CB column blocks over NK stages, each accumulator
// one chain over k in order. The next stage's operands are read while a stage is
// multiplied, and no further ahead: the weights leave few registers.
template <int NK, int CB>
__device__ __forceinline__ void multiply(f32x4 (&acc)[CB], const Operand& x, const u32x4 (&b)[CB * NK][2]) {
  u32x4 a[2][2];
  auto read = [&](int s) {
#pragma unroll
    for (int ks = 0; ks < 2; ks++) a[s & 1][ks] = x.at(ks, 128 * s);
  };
  read(0);
#pragma unroll
  for (int s = 0; s < NK; s++) {
    if (s + 1 < NK) read(s + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int c = 0; c < CB; c++) acc[c] = mfma_16x16x32(a[s & 1][ks], b[c * NK + s][ks], acc[c]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// RMSNorm in place of the tile's rows (K = 1024), two rows of a wave at a time, as rmsnorm_rows
__device__ __forceinline__ void norm_rows(uint8_t* lds, const u32x4 (&wc)[2], int wv, int lane) {
  float w[2][8];
  unpack8(wc[0], w[0]);
  unpack8(wc[1], w[1]);
  float f[2][2][8], ss[2];
  uint8_t* p[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = 2 * wv + i;
#pragma unroll
    for (int hh = 0; hh < 2; hh++) p[i][hh] = lds + r * 2 * H + 16 * ((64 * hh + lane) ^ (r & 7));
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    ss[i] = 0.f;
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
      unpack8(lds16(p[i][hh]), f[i][hh]);
#pragma unroll
      for (int e = 0; e < 8; e++) ss[i] = fmaf(f[i][hh][e], f[i][hh][e], ss[i]);
    }
  }
  wave_sum_n(ss);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const float rstd = 1.0f / sqrtf(ss[i] * (1.0f / H) + EPS);
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t n = pack_bf2(f[i][hh][2 * e] * rstd, f[i][hh][2 * e + 1] * rstd);
        o[e] = pack_bf2(w[hh][2 * e] * bflo(n), w[hh][2 * e + 1] * bfhi(n));
      }
      *reinterpret_cast<u32x4*>(p[i][hh]) = o;
    }
  }
}

// Polls are bounded: after POLL_LIMIT rounds a wave sets the launch's dead word, every wait gives up,
// and the launch's result says so (the word is its own: launches that overlap do not share it).
__device__ __noinline__ bool give_up(const Buf& sb, uint32_t spins) {
  if (sb.ld1(4u * SY_DEAD) != 0) return true;
  if (spins <= POLL_LIMIT) return false;
  sb.st1(1u, 4u * SY_DEAD);
  return true;
}
// One wave waits until the words of `lb` at `word` (its own in each lane with `mine`) have reached
// `want`: words of this XCD, stored plainly and read with non-temporal loads served by its L2, or
// (ANY) words of every XCD at device scope. False: given up.
template <bool ANY>
__device__ __forceinline__ bool wait_local(const Buf& lb, const Buf& sb, int word, bool mine, uint32_t want) {
  for (uint32_t spins = 1;; spins++) {
    const uint32_t v = mine ? __builtin_amdgcn_raw_buffer_load_b32(lb.r, 4 * word, 0, ANY ? SC1 : 2 /* nt */) : want;
    if (__ballot((int)(v - want) < 0) == 0) return true;
    if (ANY) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");  // (every round loads)
    if ((spins & 1023u) == 0 && give_up(sb, spins)) return false;
  }
}
// The same for the eight XCDs' words of a line of `sb`
__device__ __forceinline__ bool wait_xcds(const Buf& sb, int word, uint32_t want, int lane) {
  for (uint32_t spins = 1;; spins++) {
    const uint32_t v = sb.ld1(4u * (uint32_t)(word + (lane & (NXCD - 1))));
    if (__ballot((int)(v - want) < 0) == 0) return true;
    asm volatile("" ::: "memory");  // (every round loads)
    if ((spins & 1023u) == 0 && give_up(sb, spins)) return false;
  }
}
template <bool ANY>
__device__ __forceinline__ void store_local(const Buf& lb, int word, uint32_t v) {
  __builtin_amdgcn_raw_buffer_store_b32(v, lb.r, 4 * word, 0, ANY ? SC1 : 0);
}

// The launch's mode, settled once: one wave of the first workgroup on each XCD waits until every
// XCD has two workgroups of the launch, or until `ticks` have passed, and the first of them to
// know writes the word.
__device__ __forceinline__ uint32_t settle_mode(const Buf& sb, uint32_t* sync, uint64_t ticks, int lane) {
  const uint64_t t0 = wall_clock64();
  for (;;) {
    const uint32_t roles = sb.ld1(4u * (uint32_t)(32 * (lane & (NXCD - 1)) + SY_ROLE));
    const bool late = wall_clock64() - t0 >= ticks;
    if (late || __ballot(roles < 2u) == 0) {
      uint32_t m = 0u;
      if (lane == 0 && __hip_atomic_compare_exchange_strong(sync + SY_MODE, &m, late ? MODE_ANY : MODE_XCD,
                                                            __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT))
        m = late ? MODE_ANY : MODE_XCD;
      return __builtin_amdgcn_readfirstlane(m);
    }
    asm volatile("" ::: "memory");  // (every round loads)
  }
}
// The other workgroups' wait for it (0: given up)
__device__ __forceinline__ uint32_t wait_mode(const Buf& sb) {
  for (uint32_t spins = 1;; spins++) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(sb.ld1(4u * SY_MODE));
    if (m != 0u) return m;
    asm volatile("" ::: "memory");  // (every round loads)
    if ((spins & 1023u) == 0 && give_up(sb, spins)) return 0u;
  }
}

// The relay workgroup of an XCD: each wave follows G row blocks through their steps, layer by layer.
// When this XCD's tasks of the step are done for them it tells the other XCDs (one word a
// step, wave and XCD), and when all XCDs' are done it tells its own workgroups. So a word that
// crosses XCDs has one writer and eight readers; with every task storing a device-scope flag of
// its own and every waiting workgroup polling them, a hand-over took 1.5-4 us (16 tokens).
__device__ __forceinline__ void relay(const Buf& sb, const Buf& lb, const Sync& F, int nb, int G, int layers, int wv,
                                      int lane) {
  const int rb = wv * G, blocks = min(G, nb - rb);
  if (blocks <= 0) return;
  for (int l = 1; l <= layers; l++)
#pragma unroll 1
    for (int s = 0; s < NSTEP; s++) {
      int word, n;
      if (s == S_ATT) word = F.att + rb * NATT, n = NATT * blocks;
      else if (s == S_O) word = F.o + rb * NO, n = NO * blocks;
      else if (s == S_GU) word = F.gu + rb * NGU, n = NGU * blocks;
      else word = F.down + rb * ND, n = ND * blocks;
      if (!wait_local<false>(lb, sb, word + lane, lane < n, (uint32_t)l)) return;
      const int line = F.steps + (s * NW + wv) * SY_LINE;
      if (lane == 0) sb.st1((uint32_t)l, 4u * (uint32_t)line);
      if (!wait_xcds(sb, line & ~(SY_LINE - 1), (uint32_t)l, lane)) return;
      if (lane == 0) store_local<false>(lb, F.relay + s * NW + wv, (uint32_t)l);
    }
}

// Embedding rows of the prompt, and the sync area cleared for the launch that follows.
__global__ void __launch_bounds__(128) embed_rows_sync(const int* ids, const uint16_t* emb, uint16_t* h, uint32_t* err,
                                                       uint32_t* sync, int nsync, uint32_t* local, int nlocal,
                                                       uint32_t dead) {
  embed_row(ids, emb, h, err, blockIdx.x, threadIdx.x);
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < nsync; i += 128) sync[i] = i == SY_DEAD ? dead : 0u;
    for (int i = threadIdx.x; i < nlocal; i += 128) local[i] = 0u;
  }
}

constexpr int MAXK = SHORT_MAX_S;             // keys of the longest prompt
constexpr int SC_PITCH = MAXK + 4;            // score row pitch (floats); the row's probabilities overlay it
constexpr int V_OFF = 0, SC_OFF = MAXK * 256; // attention LDS: V rows, then the score rows, then the output tile
constexpr int AO_OFF = SC_OFF + 16 * SC_PITCH * 4;
constexpr int EPI_OFF = 96 * 1024;            // epilogue tiles, past every activation tile
static_assert(AO_OFF + 16 * HD * 2 <= LDS_BYTES, "attention LDS");
__device__ __forceinline__ uint32_t v_off(int row, int chunk) { return row * 256 + 16 * (chunk ^ (row & 15)); }

struct Shared {
  __align__(16) uint8_t lds[LDS_BYTES];
  float l[16];
  uint32_t ticket, ok;
};

__device__ __forceinline__ uint32_t take(uint32_t* word) {
  return __hip_atomic_fetch_add(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A workgroup's tasks: those of XCD g's list that fall to it, or (ANY) of the single list, whose
// task t is task t / 8 of XCD t % 8's. False if a wait was given up or, with a list per XCD, if the
// launch's mode is the other one (nothing has been published then: a workgroup looks before
// the first task it finishes). From the single list a task is one row block and waits before it
// loads its weights: with the weights in registers across a wait on eight XCDs' flags the
// compiler spills (211 registers), and this path is there to finish, not for speed.
template <bool ANY>
__device__ __forceinline__ bool run_tasks(const ShortArgs& P, Shared& sm, int g, int wv) {
  uint8_t* const lds = sm.lds;
  float* const s_l = sm.l;
  const int S = P.S, nb = (S + 15) / 16;
  // G consecutive row blocks to a relay wave. A task of the four products loads its weights once
  // and takes row blocks rb, rb + nq, ..: the blocks below nq run a layer's steps together, the
  // next nq behind them (consecutive blocks to a task would make the attention of the later
  // blocks, which reads all earlier rows, wait for the last round of every qkv task)
  const int G = (nb + NW - 1) / NW, nq = ANY ? nb : P.groups;
  Sync F(nb, g);
  const Buf sb(P.sync), lb(P.local);
  const int n_qkv = NQKV * nq, n_att = NATT * nb, n_o = NO * nq, n_gu = NGU * nq, n_d = ND * nq;
  const int per_layer = n_qkv + n_att + n_o + n_gu + n_d, total = per_layer * P.num_layers;
  uint8_t* ring = lds + wv * RING * STAGE;
  uint32_t* const tickets = P.sync + (ANY ? SY_ANY : 32 * g);
  bool placed = ANY, ok = true;  // placed: the mode has been looked at (wave 0)

  __syncthreads();
  if (threadIdx.x == 0) sm.ticket = take(tickets);
  for (;;) {
    // (opaque, so that the tasks' address arithmetic is not hoisted out of this loop into
    // registers that the weights need)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (ANY) asm volatile("" : "+s"(wv));  // (likewise)
    const int lane = tid & 63, r16 = lane & 15, kg = lane >> 4, rq = 4 * kg;
    __syncthreads();
    uint32_t t = __builtin_amdgcn_readfirstlane(sm.ticket);
    if (ANY) {
      g = (int)(t & (NXCD - 1));
      t >>= 3;
      F = Sync(nb, g);
    }
    if (t >= (uint32_t)total) break;
    const int l = (int)t / per_layer;
    int i = (int)t % per_layer;
    const PrefillLayerWeights& W = P.lw[l];
    const uint32_t done = (uint32_t)l + 1u;  // flag value of this layer's tasks
    auto bf = [](const void* p) { return static_cast<const uint16_t*>(p); };
    // every wave is done loading weights, and the tasks this one reads from are done
    auto ready = [&](int word, bool mine, uint32_t want) {
      if (wv == 0) {
        if (!placed) placed = wait_mode(sb) == MODE_XCD;
        const bool r = placed && wait_local<ANY>(lb, sb, word, mine, want);
        if (lane == 0) sm.ok = r;
      }
      __syncthreads();
      ok = __builtin_amdgcn_readfirstlane(sm.ok) != 0;
    };
    // ... where those are all XCDs' tasks of a step and row block: this XCD's relay word, or (ANY)
    // the tasks' flags themselves, lane 8 j + x task j of XCD x
    auto relayed = [&](int step, int rb, uint32_t want) {
      if constexpr (ANY) {
        const int ln = lane, j = ln >> 3;
        const Sync X(nb, ln & (NXCD - 1));
        const int n = step == S_ATT ? NATT : step == S_O ? NO : step == S_GU ? NGU : ND;
        const int base = step == S_ATT ? X.att : step == S_O ? X.o : step == S_GU ? X.gu : X.down;
        ready(base + n * rb + j, j < n, want);
      } else {
        ready(F.relay + step * NW + rb / G, (threadIdx.x & 63) == 0, want);
      }
    };
    // the stores of the task's row block are complete, then its flag
    auto finish = [&](int flag) {
      wait_vmem();
      __syncthreads();
      if (threadIdx.x == 0) store_local<ANY>(lb, flag, done);
    };

    if (i < n_qkv) {
      // ---------------------------------------------------------------- q, k or v head
      const int j = i % NQKV, rb0 = i / NQKV;  // j: q heads 2g, 2g + 1, k, v
      const uint16_t* wp = j < 2 ? bf(W.q_proj_weight) + (size_t)(2 * g + j) * HD * H
                                 : bf(j == 2 ? W.k_proj_weight : W.v_proj_weight) + (size_t)g * HD * H;
      u32x4 b[16][2];
      if (ANY) {
        relayed(S_DOWN, rb0, (uint32_t)l);
        if (!ok) break;
      }
      load_weights(b, wp + (size_t)16 * wv * H, H, [](int s) { return 64 * s; }, ring, lane);
      const uint16_t* nw = bf(W.input_layernorm_weight);
      const u32x4 wc[2] = {ldw(nw + 8 * lane), ldw(nw + 512 + 8 * lane)};
      // the epilogue's operands: 32 lanes a row, lane p of them dims 2p, 2p + 1 and 64 + 2p, + 1
      const int er = tid >> 5, ed = 2 * (tid & 31);
      const uint16_t* nwp = bf(j < 2 ? W.q_norm_weight : W.k_norm_weight);
      const uint32_t nw1 = ldw1(nwp + ed), nw2 = ldw1(nwp + 64 + ed);
      const size_t kvl = ((size_t)l * NKV + g) * P.max_seq * HD;
      const Buf out(j < 2 ? P.q + (2 * g + j) * HD : (j == 2 ? P.kc : P.vc) + kvl);
#pragma unroll 1
      for (int rb = rb0; rb < (ANY ? rb0 + 1 : nb); rb += nq) {
        const int tk = 16 * rb + er;
        const size_t ct = (size_t)min(tk, S - 1) * HD + ed;
        const uint32_t c1 = ldw1(P.cos_t + ct), c2 = ldw1(P.cos_t + ct + 64);
        const uint32_t s1 = ldw1(P.sin_t + ct), s2 = ldw1(P.sin_t + ct + 64);
        if (ANY) __syncthreads();  // every wave is done loading weights
        else relayed(S_DOWN, rb, (uint32_t)l);
        if (!ok) break;
        load_rows<H, 16>(P.h, 16 * rb, S, lds, wv, lane);
        __syncthreads();
        norm_rows(lds, wc, wv, lane);
        __syncthreads();
        const Operand x(lds, 2 * H, r16, kg);
        f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        multiply<16>(acc, x, b);
        // QK-norm and RoPE as in mq_prefill.hip's one-head epilogue: the sum of squares is the
        // same tree (pairs d, d + 64; eight consecutive d; then the eight groups), over 32 lanes a row
        constexpr int QP = HD + 4;
        float* tile = reinterpret_cast<float*>(lds + EPI_OFF);
#pragma unroll
        for (int e = 0; e < 4; e++) tile[(rq + e) * QP + 16 * wv + r16] = rbf(acc[0][e]);
        __syncthreads();
        const float* y = tile + er * QP + ed;
        const float x1[2] = {y[0], y[1]}, x2[2] = {y[64], y[65]};
        uint32_t o1 = pack_bf2(x1[0], x1[1]), o2 = pack_bf2(x2[0], x2[1]);
        if (j < 3) {
          float ss = (x1[0] * x1[0] + x2[0] * x2[0]) + (x1[1] * x1[1] + x2[1] * x2[1]);
          ss += dpp<0xB1>(ss);
          ss += dpp<0x4E>(ss);
          ss += dpp<0x141>(ss);
          ss += dpp<0x140>(ss);
          const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
          ss = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
          const float rstd = 1.0f / sqrtf(ss * (1.0f / HD) + EPS);
          const uint32_t a1 = pack_bf2(x1[0] * rstd, x1[1] * rstd), a2 = pack_bf2(x2[0] * rstd, x2[1] * rstd);
          const uint32_t n1 = pack_bf2(bflo(nw1) * bflo(a1), bfhi(nw1) * bfhi(a1));
          const uint32_t n2 = pack_bf2(bflo(nw2) * bflo(a2), bfhi(nw2) * bfhi(a2));
          o1 = pack_bf2(rbf(bflo(n1) * bflo(c1)) - rbf(bflo(n2) * bflo(s1)),
                        rbf(bfhi(n1) * bfhi(c1)) - rbf(bfhi(n2) * bfhi(s1)));
          o2 = pack_bf2(rbf(bflo(n2) * bflo(c2)) + rbf(bflo(n1) * bflo(s2)),
                        rbf(bfhi(n2) * bfhi(c2)) + rbf(bfhi(n1) * bfhi(s2)));
        }
        if (tk < S) {
          // (with a list per XCD read by this XCD alone: plain stores)
          const uint32_t o = 2u * (uint32_t)((j < 2 ? QS : HD) * tk + ed);
          __builtin_amdgcn_raw_buffer_store_b32(o1, out.r, o, 0, ANY ? SC1 : 0);
          __builtin_amdgcn_raw_buffer_store_b32(o2, out.r, o + 128u, 0, ANY ? SC1 : 0);
        }
        finish(F.qkv + NQKV * rb + j);
      }
      if (!ok) break;
    } else if ((i -= n_qkv) < n_att) {
      // ---------------------------------------------------------------- attention
      const int qb = i >> 1, hh = i & 1, h = 2 * g + hh, r0 = 16 * qb;
      const int nk = min(S, r0 + 16), nk32 = (nk + 31) & ~31;
      // this head's q rows of the query block, and the k and v rows of every block up to it
      const int jt = lane & 3;
      ready(F.qkv + lane, (lane >> 2) <= qb && (jt >= 2 || ((lane >> 2) == qb && jt == hh)),
            done);
      if (!ok) break;
      const size_t kvl = ((size_t)l * NKV + g) * P.max_seq * HD;
      const Buf qbuf(P.q + h * HD), kbuf(P.kc + kvl);
      // V rows (past the block's last key: that key again, times probability 0)
      const uint16_t* V = P.vc + kvl;
      for (int n = wv; n < nk32 / 4; n += NW) {
        const int row = 4 * n + (lane >> 4), chunk = (lane & 15) ^ (row & 15);
        const uint32_t src = 2u * (uint32_t)(min(row, nk - 1) * HD + 8 * chunk);
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_addr(lds) + V_OFF + 1024u * (uint32_t)n);
        if (ANY) dma16_at_sc1(V, src, dst);
        else dma16_at_nt(V, src, dst);
      }
      u32x4 qf[4];
#pragma unroll
      for (int ks = 0; ks < 4; ks++)
        qf[ks] = ld4_xcd<ANY>(qbuf, 2u * (uint32_t)(min(r0 + r16, S - 1) * QS + 32 * ks + 8 * kg));
      float* sc = reinterpret_cast<float*>(lds + SC_OFF);
      constexpr int KT = MAXK / (16 * NW);  // key tiles a wave
      u32x4 kf[KT][4];
#pragma unroll
      for (int n = 0; n < KT; n++) {
        const int k0 = 16 * (wv + NW * n);
        if (k0 < nk)
#pragma unroll
          for (int ks = 0; ks < 4; ks++)
            kf[n][ks] = ld4_xcd<ANY>(kbuf, 2u * (uint32_t)(min(k0 + r16, nk - 1) * HD + 32 * ks + 8 * kg));
      }
#pragma unroll
      for (int n = 0; n < KT; n++) {
        const int k0 = 16 * (wv + NW * n), key = k0 + r16;
        if (k0 < nk) {
          f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 4; ks++) a = mfma_16x16x32(qf[ks], kf[n][ks], a);
#pragma unroll
          for (int e = 0; e < 4; e++)
            sc[(rq + e) * SC_PITCH + key] = (key <= r0 + rq + e && key < nk) ? a[e] * P.scale : -INFINITY;
        }
      }
      wait_vm<0>();  // this wave's V rows
      __syncthreads();
      {
        constexpr int NU = MAXK / 64;
        const int nu = (nk + 63) >> 6;
        float x[2][NU], mx[2], sum[2];
#pragma unroll
        for (int r = 0; r < 2; r++) {
          mx[r] = -INFINITY;
#pragma unroll
          for (int u = 0; u < NU; u++) {
            x[r][u] = u < nu ? sc[(2 * wv + r) * SC_PITCH + lane + 64 * u] : -INFINITY;
            mx[r] = fmaxf(mx[r], lane + 64 * u < nk ? x[r][u] : -INFINITY);
          }
        }
        wave_max_n(mx);
#pragma unroll
        for (int r = 0; r < 2; r++) {
          // the row's probabilities overlay its scores (which this wave alone reads, above)
          uint16_t* pr = reinterpret_cast<uint16_t*>(sc + (2 * wv + r) * SC_PITCH);
          sum[r] = 0.f;
#pragma unroll
          for (int u = 0; u < NU; u++) {
            if (u >= nu) break;
            const float ev = exp_fast(x[r][u] - mx[r]);  // (a row's own key is never masked: its maximum is finite)
            const float e = lane + 64 * u < nk ? ev : 0.f;
            sum[r] += e;
            pr[lane + 64 * u] = (uint16_t)f2bf(e);
          }
        }
        wave_sum_n(sum);
        if (lane == 0) {
          s_l[2 * wv] = sum[0];
          s_l[2 * wv + 1] = sum[1];
        }
      }
      __syncthreads();
      // P.V: wave wv owns dims 16 wv .. 16 wv + 15
      typedef short v4s __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4s lds_v4s;
      const uint32_t vb = lds_addr(lds) + V_OFF;
      f32x4 oacc = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int k0 = 0; k0 < nk32; k0 += 32) {
        const int ra = k0 + 8 * kg + (r16 >> 2), dq = 16 * wv + 4 * (r16 & 3);
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(uintptr_t)(vb + v_off(ra, dq >> 3) + 2 * (dq & 7)));
        const v4s hi =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(uintptr_t)(vb + v_off(ra + 4, dq >> 3) + 2 * (dq & 7)));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        const u32x4 pf = lds16(reinterpret_cast<const uint8_t*>(sc + r16 * SC_PITCH) + 2 * (k0 + 8 * kg));
        oacc = mfma_16x16x32(pf, u32x4{l2.x, l2.y, h2.x, h2.y}, oacc);
      }
      uint16_t* ot = reinterpret_cast<uint16_t*>(lds + AO_OFF);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float inv = 1.0f / s_l[rq + e];
        ot[(rq + e) * HD + 16 * wv + r16] = (uint16_t)f2bf(oacc[e] * inv);
      }
      __syncthreads();
      if (tid < 256) {
        const int r = tid >> 4, c = tid & 15;
        if (r0 + r < S) {
          const Buf out(P.att + h * HD);
          out.st4(lds16(lds + AO_OFF + r * HD * 2 + 16 * c), 2u * (uint32_t)((r0 + r) * QS + 8 * c));
        }
      }
      finish(F.att + NATT * qb + hh);
    } else if ((i -= n_att) < n_o || (i - n_o >= n_gu)) {
      // ---------------------------------------------------------------- o_proj or down_proj
      // The k quarters are chains of their own, one or two column blocks to a wave, added in
      // order in the epilogue, which rounds the Linear output and adds the residual
      auto residual = [&](auto oc) {
        constexpr bool O = decltype(oc)::value;
        constexpr int K = O ? QS : I, CB = O ? 2 : 1, TC = 32 * CB, KQ = K / 4, NK = KQ / 64, TP = TC + 4;
        constexpr int NC = O ? NO : ND;
        const int n = O ? i : i - n_o - n_gu, ct = NC * g + n % NC, rb0 = n / NC;
        const int z = wv & 3, cb0 = CB * (wv >> 2);  // k quarter, first column block
        u32x4 b[CB * NK][2];
        if (ANY) {
          relayed(O ? S_ATT : S_GU, rb0, done);
          if (!ok) return;
        }
        load_weights(b, bf(O ? W.o_proj_weight : W.down_proj_weight) + (size_t)(TC * ct + 16 * cb0) * K + KQ * z, K,
                     [](int s) { return (s / NK) * 16 * K + 64 * (s % NK); }, ring, lane);
        const Buf hb(P.h + TC * ct);
        const int er = tid / (TC / 2), ec = 2 * (tid % (TC / 2));
        const bool mine = tid < 8 * TC;  // two columns a thread
#pragma unroll 1
        for (int rb = rb0; rb < (ANY ? rb0 + 1 : nb); rb += nq) {
          if (ANY) __syncthreads();
          else relayed(O ? S_ATT : S_GU, rb, done);
          if (!ok) return;
          // the residual rows (their last writers are done: the qkv or gu tasks of these rows read them)
          const int row = 16 * rb + er;
          uint32_t hr = 0u;
          if (mine) hr = hb.ld1(2u * (uint32_t)(min(row, S - 1) * H + ec));
          load_rows<K, 16>(O ? P.att : P.mid, 16 * rb, S, lds, wv, lane);
          __syncthreads();
          const Operand x(lds + 2 * KQ * z, 2 * K, r16, kg);
          f32x4 acc[CB];
#pragma unroll
          for (int c = 0; c < CB; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
          multiply<NK>(acc, x, b);
          float* part = reinterpret_cast<float*>(lds + EPI_OFF);  // [quarter][16][TP]
#pragma unroll
          for (int c = 0; c < CB; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) part[(16 * z + rq + e) * TP + 16 * (cb0 + c) + r16] = acc[c][e];
          __syncthreads();
          if (mine) {
            float f[2] = {part[er * TP + ec], part[er * TP + ec + 1]};
#pragma unroll
            for (int q = 1; q < 4; q++)
#pragma unroll
              for (int e = 0; e < 2; e++) f[e] += part[(16 * q + er) * TP + ec + e];
            if (row < S) hb.st1(pack_bf2(bflo(hr) + rbf(f[0]), bfhi(hr) + rbf(f[1])), 2u * (uint32_t)(row * H + ec));
          }
          finish((O ? F.o : F.down) + NC * rb + n % NC);
        }
      };
      if (i < n_o) residual(std::true_type{});
      else residual(std::false_type{});
      if (!ok) break;
    } else {
      // ---------------------------------------------------------------- gate/up
      i -= n_o;
      const int ct = NGU * g + i % NGU, rb0 = i / NGU;
      // waves 0..3: gate blocks of 16 units, waves 4..7: their up blocks
      const int ub = wv & 3;
      u32x4 b[16][2];
      if (ANY) {
        relayed(S_O, rb0, done);
        if (!ok) break;
      }
      load_weights(b, bf(wv < 4 ? W.gate_proj_weight : W.up_proj_weight) + (size_t)(64 * ct + 16 * ub) * H, H,
                   [](int s) { return 64 * s; }, ring, lane);
      const uint16_t* nw = bf(W.post_attn_layernorm_weight);
      const u32x4 wc[2] = {ldw(nw + 8 * lane), ldw(nw + 512 + 8 * lane)};
      const Buf out(P.mid + 64 * ct);
#pragma unroll 1
      for (int rb = rb0; rb < (ANY ? rb0 + 1 : nb); rb += nq) {
        if (ANY) __syncthreads();
        else relayed(S_O, rb, done);
        if (!ok) break;
        load_rows<H, 16>(P.h, 16 * rb, S, lds, wv, lane);
        __syncthreads();
        norm_rows(lds, wc, wv, lane);
        __syncthreads();
        const Operand x(lds, 2 * H, r16, kg);
        f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        multiply<16>(acc, x, b);
        constexpr int UP = 64 + 4;  // tile pitch (floats): gate rows, then up rows
        float* tile = reinterpret_cast<float*>(lds + EPI_OFF);
#pragma unroll
        for (int e = 0; e < 4; e++) tile[((wv < 4 ? 0 : 16) + rq + e) * UP + 16 * ub + r16] = rbf(acc[0][e]);
        __syncthreads();
        const int er = tid >> 5, ec = 2 * (tid & 31), row = 16 * rb + er;  // two units a thread
        const float* gr = tile + er * UP + ec;
        const float* ur = gr + 16 * UP;
        const float g0 = gr[0], g1 = gr[1];
        const float s0 = rbf(g0 / (1.0f + expf(-g0))), s1 = rbf(g1 / (1.0f + expf(-g1)));
        if (row < S) out.st1(pack_bf2(s0 * ur[0], s1 * ur[1]), 2u * (uint32_t)(row * I + ec));
        finish(F.gu + NGU * rb + i % NGU);
      }
      if (!ok) break;
    }
    // (not earlier: a ticket held while its workgroup waits is a task that no one prepares)
    if (tid == 0) sm.ticket = take(tickets);
  }
  return ok;
}

__global__ void __launch_bounds__(NT) prefill_short(ShortArgs P) {
  __shared__ Shared sm;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  const int g = (int)(xcc & (NXCD - 1));  // this XCD's KV group and column slices
  const Buf sb(P.sync);
  // the XCD's first workgroup is its relay
  if (threadIdx.x == 0) sm.ticket = take(P.sync + 32 * g + SY_ROLE);
  __syncthreads();
  const bool first = __builtin_amdgcn_readfirstlane(sm.ticket) == 0;
  if (!first && run_tasks<false>(P, sm, g, wv)) return;
  __syncthreads();
  if (wv == 0) {
    const uint32_t m = first ? settle_mode(sb, P.sync, P.place_ticks, threadIdx.x & 63) : wait_mode(sb);
    if (threadIdx.x == 0) sm.ok = m;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(sm.ok) == MODE_ANY) {
    run_tasks<true>(P, sm, 0, wv);
  } else if (first) {
    const int nb = (P.S + 15) / 16;
    relay(sb, Buf(P.local), Sync(nb, g), nb, (nb + NW - 1) / NW, P.num_layers, wv, threadIdx.x & 63);
  }
}

}  // namespace ps

int prefill_short_run(const int* ids, const uint16_t* embed, const ps::ShortArgs& A, int debug, hipStream_t stream) {
  const int nb = (A.S + 15) / 16;
  ps::embed_rows_sync<<<A.S, 128, 0, stream>>>(ids, embed, A.h, A.err, A.sync, ps::SYNC_WORDS, A.local,
                                               ps::NXCD * ps::local_words(nb), debug & MQ_DEBUG_PREFILL_GAVE_UP ? 1u : 0u);
  if (hipGetLastError() != hipSuccess) return MQ_ERR_HIP;
  ps::ShortArgs B = A;
  B.groups = nb < ps::GROUPS ? nb : ps::GROUPS;
  B.place_ticks = debug & MQ_DEBUG_PREFILL_ANY_XCD ? 0 : ps::PLACE_TICKS;
  ps::prefill_short<<<ps::NWG, ps::NT, 0, stream>>>(B);
  return hipGetLastError() == hipSuccess ? MQ_OK : MQ_ERR_HIP;
}

}  // namespace mq
