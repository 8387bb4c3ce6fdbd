// Tiled matrix-core GEMM for any operand orientation and any (ragged) M, N, K:
//   C[m, n] = sum_k A(m, k) B(n, k),   fp32 accumulation,
// where each operand is stored either with k contiguous (rows of k: activations X, a weight W in X W^T)
// or with its own index contiguous ("K-major": dY and X in dW = dY^T X, W in dX = dY W).  Nothing is
// re-laid out in memory: a K-major tile is read through the gfx950 LDS transpose read.
//
// Bound by the matrix cores once 256 x 256 tiles fill the CUs, by the weight stream below a few hundred rows.
//  * Schedule: v_mfma_f32_16x16x32, a ring of 64-wide k-tiles filled by wave-wide direct-to-LDS loads, fragment
//    reads one k-step ahead, refills and reads spread through the MFMAs.  8192 x 12288 x 4096 (bf16): k-contiguous
//    operands 596 us (1384 TFLOP/s), K-major B 594, both K-major 599; with the transposed copies made first the
//    K-major forms cost 24 us per 8192 x 4096 operand more, and a token count off the 8-element grid had no
//    matrix-core path at all (333 tokens, 4096 x 4096 weight gradient: 390 us, here 20).
//  * Range-checked buffer loads make every tile straight-line code: ragged rows and k read zeros, prefetches past
//    the end fetch nothing.  The descriptors of the next k-tile are scalar work placed between the MFMAs of the
//    step before (formed after the barrier instead: 3-7 % slower), in 32-bit units of 16 bytes (64-bit clamps
//    became vector compares and per-lane descriptor loops: 15 % slower).
#pragma once
#include <type_traits>

#include "common.h"

namespace q3gemm {

// Workgroup barrier for a direct-to-LDS ring: this wave's loads older than its newest N have landed in
// LDS and its own LDS reads are done (vmcnt(N) lgkmcnt(0)), then s_barrier.  __syncthreads() would drain
// every prefetched stage of the ring at each k-tile.
template <int N> Q3_DEV void ring_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (0 << 8));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
Q3_DEV void lds_wait() { __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14)); }  // lgkmcnt(0)

// LDS image of one operand's [BD][64] tile.
//  * k contiguous: 128-byte rows, 8 rows per wave-wide 1 KB load, 16-byte chunk c of row r at c ^ (r & 7):
//    fragment reads (16 rows at one chunk) are conflict free.
//  * K-major: BD contiguous elements per k, 512 / BD k-rows per wave-wide load ("slot" s holds the k-rows
//    s, s + BD / 8, s + 2 BD / 8, ...).  Slots start at 1056 s + 128 (s / 8): four consecutive k-rows sit
//    32 bytes apart modulo the 256-byte bank span and k + 8 another 128 bytes away, so the 32 lanes of half a
//    transpose read (two groups of 4 k-rows x 32 bytes) touch every bank once.
constexpr int slot_base(int s) { return s * 1056 + (s >> 3) * 128; }
template <int BD, bool KM> constexpr int tile_bytes() {
  return KM ? (slot_base(BD / 8) + 15) / 16 * 16 : BD * 128;
}
constexpr int kSlot4 = 4 * 1056;  // distance of k + 4 (4 slots that never straddle a multiple of 8)

struct Operand {
  const u16* p[3];
  int64_t ld[3];
};

struct Args {
  Operand a, b;
  int64_t M, N, K;       // N: rows of the B operand (both weights of a gate/up pair)
  int axis, pieces;      // 0: one piece; 1: A and B in pieces along K; 2: B and C along N; 3: A and C along M
  int64_t len[3];        // lengths of the pieces along that axis: every piece starts a tile (a k-tile) of its own
  int tms, tns;          // tile rows and columns of this launch
  int splits;            // K splits; > 1: fp32 partial products at part + split * M * N
  float* part;
  void* c[3];
  int64_t ldc[3];
  int vec;               // C rows take 16-byte stores
  const u16* res;        // C = res + round(product)
  int64_t ldres;
  // gate/up pair: G, U stored when set (c[0] = Y); backward: g / u inputs, dg = c[0], du = c[1]
  u16 *g, *u;
  const u16 *gin, *uin;
  int64_t ldgu;
  // cross-entropy statistics (c[0] takes the logits): target columns, partials [group][ldp]
  const int64_t* tgt;
  float *m_part, *s_part, *pick;
  int64_t part0, ldp, col0;
};

// Work item -> (tile, split): each XCD (workgroup ids congruent mod 8) takes a contiguous range of items,
// splits outermost, so its L2 holds one k-range of the shared operand; tiles in groups of 4 tile-rows.
Q3_DEV void work_coords(int bid, int tiles_m, int tiles_n, int splits, int& tm, int& tn, int& sp) {
  constexpr int GROUP = 4;
  const int tiles = tiles_m * tiles_n, total = tiles * splits;
  const int xcd = bid & 7, per = total >> 3, rem = total & 7;
  int w = xcd * per + min(xcd, rem) + (bid >> 3);
  sp = w / tiles;
  w -= sp * tiles;
  const int width = GROUP * tiles_n;
  const int first = (w / width) * GROUP;
  const int gsize = min(tiles_m - first, GROUP);
  tm = first + (w % width) % gsize;
  tn = (w % width) / gsize;
}

// EPI 0: plain / residual / split partials; 2: cross-entropy statistics (per row and 128-column group: the max and the
// sum of exp(z - max) to m_part / s_part [part0 + group][row], the logit of column tgt[row] - col0 to pick[row]) of
// the rounded logits, which are stored too; 3: gate/up SwiGLU; 5: SwiGLU backward.  KP: A and B in pieces along K.
template <typename T, int BM, int BN, int WM, int WN, int STAGES, bool AT, bool BT, int EPI, bool KP>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tile_kernel(Args ar) {
  constexpr int NW = WM * WN;
  constexpr int TMW = BM / WM, TNW = BN / WN, FM = TMW / 16, FN = TNW / 16;
  constexpr int AL = BM / 8, BL = BN / 8;  // wave-wide 1 KB loads per operand and k-tile
  static_assert(AL % NW == 0 && BL % NW == 0, "loads must split evenly over the waves");
  static_assert(STAGES >= 2 && STAGES <= 4, "ring depth");
  static_assert(TMW % 16 == 0 && TNW % 16 == 0, "fragments");
  static_assert(!AT || (BM == 64 || BM == 128 || BM == 256), "K-major slots");
  static_assert(!BT || (BN == 64 || BN == 128 || BN == 256), "K-major slots");
  constexpr int LPW = (AL + BL) / NW, LA = AL / NW;
  constexpr int ABYTES = tile_bytes<BM, AT>(), STAGE = ABYTES + tile_bytes<BN, BT>();
  constexpr int BMAX = BM * BN * 2;
  constexpr int LDSB = STAGES * STAGE > BMAX ? STAGES * STAGE : BMAX;
  __shared__ __attribute__((aligned(1024))) char lds[LDSB];

  int tm, tn, sp;
  work_coords(blockIdx.x, ar.tms, ar.tns, ar.splits, tm, tn, sp);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int M = (int)ar.M, N = (int)ar.N;

  // this tile's pieces along M / N
  const u16 *pa = ar.a.p[0], *pb = ar.b.p[0];
  int64_t lda = ar.a.ld[0], ldb = ar.b.ld[0], ldc = ar.ldc[0];
  void* cp = ar.c[0];
  int begm = 0, begn = 0, mrows = M, ncols = N;  // the piece's first row / column, its extent
  if (ar.axis >= 2) {
    int s = 0, t = ar.axis == 2 ? tn : tm, beg = 0;
    const int bt = ar.axis == 2 ? BN : BM;
    while (s + 1 < ar.pieces && t >= ((int)ar.len[s] + bt - 1) / bt) {
      t -= ((int)ar.len[s] + bt - 1) / bt;
      beg += (int)ar.len[s++];
    }
    cp = ar.c[s];
    ldc = ar.ldc[s];
    if (ar.axis == 2) {
      pb = ar.b.p[s];
      ldb = ar.b.ld[s];
      tn = t;
      begn = beg;
      ncols = (int)ar.len[s];
    } else {
      pa = ar.a.p[s];
      lda = ar.a.ld[s];
      tm = t;
      begm = beg;
      mrows = (int)ar.len[s];
    }
  }
  // gate/up: the operand's 16-row blocks come from Wg and Wu in turn; a wave's loads (8 rows each, NW apart) are
  // all of one weight
  static_assert(EPI != 3 || NW % 4 == 0, "loads of one wave alternate weights");
  if (EPI == 3 && (wave & 2)) pb = ar.b.p[1];
  const int ma = tm * BM, nb = tn * BN;  // first row / column of the tile within its piece
  auto ktiles = [](int64_t k) { return (int)((k + 63) / 64); };
  int nk_all = ktiles(KP ? ar.len[0] : ar.K);
  if constexpr (KP)
    for (int i = 1; i < ar.pieces; ++i) nk_all += ktiles(ar.len[i]);
  const int kper = (nk_all + ar.splits - 1) / ar.splits;
  const int kt0 = sp * kper, nk = max(0, min(kper, nk_all - kt0));

  // ---- global -> LDS through range-checked buffer loads: rows past the operand's end read zeros, and a k
  // chunk past the end of a k-contiguous row is sent out of range, so every tile (ragged or past the last)
  // runs the same straight-line code.
  constexpr uint32_t kOob = 0x80000000u;
  // k contiguous: lane -> row lane / 8, logical chunk (lane % 8) ^ (row & 7); K-major: k-row and chunk of the slot
  const int achk = AT ? (lane % (BM / 8)) : ((lane & 7) ^ (lane >> 3));
  const int bchk = BT ? (lane % (BN / 8)) : ((lane & 7) ^ (lane >> 3));
  auto lane_off = [&](int64_t ld, bool km, int chk, int bd) {
    return (uint32_t)(((km ? (lane / (bd / 8)) * (bd / 8) : (lane >> 3)) * (int)ld + chk * 8) * 2);
  };
  uint32_t offa = lane_off(lda, AT, achk, BM), offb = lane_off(ldb, BT, bchk, BN);
  constexpr int BDIV = EPI == 3 ? 2 : 1;  // gate/up: each weight holds half of the operand's rows
  // The next k-tile's descriptors, formed while the matrix cores run (prep) and used after the barrier (issue).
  // They span one tile's rows, so the operand itself may be of any size.
  int64_t basea = 0, baseb = 0;  // element offset of the tile in its piece
  int rema = 0, remb = 0;        // 16-byte units: k contiguous, from there to the end of the tile's last row; K-major,
                                 // from there to the end of the piece's part of a k-row
  int krem = 0;                  // k left in the piece
  int tleft = nk;                // k-tiles left in this split
  auto start = [&](int64_t kp, int64_t k0) {  // the cursor at k0 of a piece of kp
    basea = AT ? k0 * lda + ma : (int64_t)ma * lda + k0;
    baseb = BT ? k0 * ldb + nb : (int64_t)(nb / BDIV) * ldb + k0;
    rema = AT ? (mrows - ma) >> 3 : (int)(((min(mrows - ma, BM) - 1) * lda + kp - k0) >> 3);
    remb = BT ? (ncols - nb) >> 3 : (int)(((min(ncols - nb, BN) / BDIV - 1) * ldb + kp - k0) >> 3);
    krem = (int)(kp - k0);
  };
  int pi = 0;
  auto piece = [&](int i, int64_t k0) {
    pa = ar.a.p[i];
    pb = ar.b.p[i];
    lda = ar.a.ld[i];
    ldb = ar.b.ld[i];
    offa = lane_off(lda, AT, achk, BM);
    offb = lane_off(ldb, BT, bchk, BN);
    start(ar.len[i], k0);
  };
  if constexpr (KP) {
    int t = kt0;
    while (pi + 1 < ar.pieces && t >= ktiles(ar.len[pi])) t -= ktiles(ar.len[pi++]);
    piece(pi, (int64_t)t * 64);
  } else {
    start(ar.K, (int64_t)kt0 * 64);
  }
  auto turn = [&]() {  // KP: on to the next piece once the cursor has left this one (before a k-tile's prep)
    if constexpr (KP) {
      if (krem <= 0 && pi + 1 < ar.pieces) piece(++pi, 0);
    }
  };
  typedef decltype(__builtin_amdgcn_make_buffer_rsrc((void*)nullptr, 0, 0, 0)) rsrc_t;
  rsrc_t da, db;
  uint32_t va, vb;
  auto prep = [&]() {
    // A descriptor spans at most 2^31 - 16 bytes (row strides stay below 2^22); past the last k-tile, the only
    // place where nothing is left, it is empty.
    const int krow = min(krem, 64) - 1;  // last k-row of the tile
    auto bytes = [&](int rem) { return tleft > 0 ? min(rem, 0x7ffffff) * 16 : 0; };
    const int ea = AT ? krow * (int)(lda >> 3) + rema : rema, eb = BT ? krow * (int)(ldb >> 3) + remb : remb;
    da = __builtin_amdgcn_make_buffer_rsrc((void*)(pa + basea), 0, bytes(ea), 0x00027000);
    db = __builtin_amdgcn_make_buffer_rsrc((void*)(pb + baseb), 0, bytes(eb), 0x00027000);
    va = !AT && achk * 8 >= krem ? kOob : offa;
    vb = !BT && bchk * 8 >= krem ? kOob : offb;
    krem -= 64;
    --tleft;
    basea += AT ? 64 * lda : 64;
    baseb += BT ? 64 * ldb : 64;
    if (!AT) rema -= 8;
    if (!BT) remb -= 8;
  };
  auto issue = [&](int stage) {
    char* st = lds + stage * STAGE;
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      if (i < LA) {
        const int q = wave + NW * i;  // row group of 8, or slot
        char* dst = st + (AT ? slot_base(q) : q * 1024);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(da, (__attribute__((address_space(3))) void*)dst, 16,
                                                 va + (uint32_t)(q * (AT ? 2 : 16) * (int)lda), 0, 0, 0);
      } else {
        const int q = wave + NW * (i - LA);
        char* dst = st + ABYTES + (BT ? slot_base(q) : q * 1024);
        const int rr = EPI == 3 ? ((q >> 2) * 2 + (q & 1)) * 16 : q * (BT ? 2 : 16);  // row offset x 2 bytes
        __builtin_amdgcn_raw_ptr_buffer_load_lds(db, (__attribute__((address_space(3))) void*)dst, 16,
                                                 vb + (uint32_t)(rr * (int)ldb), 0, 0, 0);
      }
    }
  };

  // ---- LDS -> fragments: lane l holds row l % 16, k = 8 (l / 16) .. + 7 of each 32-wide k-step
  const int quarter = lane >> 4, j16 = lane & 15;
  auto frag_base = [&](bool km, int bd, int first, int ks) -> uint32_t {
    if (!km) return (uint32_t)((first + j16) * 128 + (((ks * 4 + quarter) ^ (j16 & 7)) << 4));
    const int ns = bd / 8;  // slots
    const int k = 8 * quarter + (j16 >> 2);
    return (uint32_t)(slot_base(k % ns) + (k / ns) * bd * 2 + (first + 4 * (j16 & 3)) * 2);
  };
  uint32_t fa[2], fb[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    fa[ks] = frag_base(AT, BM, wm * TMW, ks) + (AT ? ks * 512 : 0);
    fb[ks] = ABYTES + frag_base(BT, BN, wn * TNW, ks) + (BT ? ks * 512 : 0);
  }
  bf16x8_t af[2][FM], bfr[2][FN];
  auto tread = [&](const char* p) { return __builtin_bit_cast(bf16x8_t, lds_frag_tr(p, kSlot4)); };
  auto load = [&](int stage, int buf, int ks) {
    const char* sb = lds + stage * STAGE;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if constexpr (AT) af[buf][i] = tread(sb + fa[ks] + i * 32);
      else af[buf][i] = *reinterpret_cast<const bf16x8_t*>(sb + fa[ks] + i * 16 * 128);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (BT) bfr[buf][j] = tread(sb + fb[ks] + j * 32);
      else bfr[buf][j] = *reinterpret_cast<const bf16x8_t*>(sb + fb[ks] + j * 16 * 128);
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int st = 0; st < STAGES - 1; ++st) {
    prep();
    issue(st);
    turn();
  }
  prep();
  ring_sync<(STAGES - 2) * LPW>();
  issue(STAGES - 1);
  load(0, 0, 0);
  constexpr int RD = FM * (AT ? 2 : 1) + FN * (BT ? 2 : 1), MF = FM * FN;  // LDS reads and MFMAs per k-step
  auto tile = [&](int stage, int next) {
    turn();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      __builtin_amdgcn_sched_barrier(0);
      if (ks == 0) {
        lds_wait();  // this step's fragments were read a step ago; keeps the LDS counter in range below
        load(stage, 1, 1);
        prep();  // the refill of the step below
      } else {
        ring_sync<(STAGES - 2) * LPW>();  // tile kt + 1 resident, every wave done with tile kt
        issue(stage);
        load(next, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma_16x16x32<T>(bfr[ks][j], af[ks][i], acc[i][j]);
      // spread the step's memory instructions through its MFMAs (refills first, two MFMAs apart where
      // there are enough of them, then the fragment reads; the other step's reads start after 3/8 of them)
      if constexpr (MF >= 16) {
        constexpr int LEAD = MF * 3 / 8;
        if (ks == 1) {
          constexpr int PER = MF >= 2 * LPW + RD / 2 ? 2 : 1;
          constexpr int LEFT = MF - PER * LPW > 0 ? MF - PER * LPW : 1, RPM = (RD + LEFT - 1) / LEFT;
#pragma unroll
          for (int q = 0; q < LPW; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
          }
#pragma unroll
          for (int q = 0; q < (RD + RPM - 1) / RPM; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
        } else {
          constexpr int LEFT = MF - LEAD, RPM = (RD + LEFT - 1) / LEFT;
#pragma unroll
          for (int q = 0; q < LEAD; ++q) {  // the next descriptors' scalar work between the leading MFMAs
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x004, 4, 0);
          }
#pragma unroll
          for (int q = 0; q < (RD + RPM - 1) / RPM; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (STAGES == 2 && !KP) {  // unrolled: the stages' LDS addresses are constants
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      tile(0, 1);
      tile(1, 0);
    }
    if (kt < nk) tile(0, 1);
  } else {
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int next = stage + 1 == STAGES ? 0 : stage + 1;
      tile(stage, next);
      stage = next;
    }
  }
  ring_sync<0>();  // every wave is done with the operand ring and no refill is in flight

  // ---- epilogue: lane owns row m (j16) and 4 consecutive columns of each 16 x 16 block
  if (ar.splits > 1) {
    float* P = ar.part + (int64_t)sp * M * N;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = ma + wm * TMW + i * 16 + j16;
      if (row < mrows) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int col = nb + wn * TNW + j * 16 + 4 * quarter;  // pieces and N are multiples of 8
          if (col < ncols) *reinterpret_cast<f32x4*>(P + (int64_t)(begm + row) * N + begn + col) = acc[i][j];
        }
      }
    }
    return;
  }
  u16* C = reinterpret_cast<u16*>(cp);
  {
    // 16-bit outputs: each wave rounds its tile into a private LDS block (16-byte chunks XOR-swizzled by row),
    // then works on whole rows with 16-byte accesses.
    if (ar.vec || EPI != 0) {
      constexpr int NC = EPI == 3 ? TNW / 2 : TNW, CH = NC / 8, RPI = 64 / CH;
      static_assert(CH == 2 || CH == 4 || CH == 8 || CH == 16, "16-byte chunks per staged row");
      char* wl = lds + wave * (TMW * NC * 2);
      auto swz = [&](int r) { return CH == 16 ? (r & 15) : CH == 8 ? ((r >> 1) & 7) : CH == 4 ? ((r >> 2) & 3) : ((r >> 3) & 1); };
      auto stage_out = [&](int i, int jc, uint32_t lo, uint32_t hi) {
        const int r = i * 16 + j16, c = (jc * 16 + 4 * quarter) >> 3;
        *reinterpret_cast<i32x2*>(wl + r * (NC * 2) + ((c ^ swz(r)) << 4) + (quarter & 1) * 8) = i32x2{(int)lo, (int)hi};
      };
      const int c = lane % CH;
      const int rlim = mrows - ma - wm * TMW;  // valid rows / columns of the wave's block
      auto row_chunk = [&](int r) { return *reinterpret_cast<const i32x4*>(wl + r * (NC * 2) + ((c ^ swz(r)) << 4)); };
      if constexpr (EPI == 2) {
        // The logits are rounded into the staged block first, so their accumulators are dead before the statistics'
        // temporaries are live; then each row's 16 chunks (16 lanes) are read once, for the store and the statistics.
        static_assert(TNW == 128 && CH == 16, "one statistics partial per wave and row");
        const int clim = ncols - nb - wn * TNW;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            stage_out(i, j, pack2<T>(acc[i][j][0], acc[i][j][1]), pack2<T>(acc[i][j][2], acc[i][j][3]));
        lds_wait();
        __builtin_amdgcn_wave_barrier();
        const int64_t part = (ar.part0 + (nb + wn * TNW) / 128) * ar.ldp;
        const int have = min(clim - c * 8, 8);  // columns of this lane's chunk
#pragma unroll 2
        for (int q = 0; q < TMW / RPI; ++q) {
          const int r = q * RPI + lane / CH;
          const int row = ma + wm * TMW + r;
          const i32x4 raw = row_chunk(r);
          Vec<T> v = unpack_vec<T>(raw);
          int64_t t = -1;
          if (r < rlim) {
            t = ar.tgt[row] - ar.col0 - (nb + wn * TNW + c * 8);  // target within the lane's chunk
            u16* dst = C + (int64_t)row * ldc + nb + wn * TNW + c * 8;
            if (have == 8) {
              *reinterpret_cast<i32x4*>(dst) = raw;
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (e < have) dst[e] = (u16)((uint32_t)raw[e >> 1] >> (16 * (e & 1)));
            }
          }
          float mx = -INFINITY;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if (e >= have) v.v[e] = -INFINITY;
            mx = fmaxf(mx, v.v[e]);
            if (e == t && e < have) ar.pick[row] = v.v[e];
          }
          mx = group_max<16>(mx);
          float sm = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) sm += mx == -INFINITY ? 0.f : __expf(v.v[e] - mx);
          sm = group_sum<16>(sm);
          if (c == 0 && r < rlim && clim > 0) {  // a wave past the last column has no partial
            ar.m_part[part + row] = mx;
            ar.s_part[part + row] = sm;
          }
        }
        return;
      } else if constexpr (EPI == 3) {
        const int64_t o0 = (int64_t)(ma + wm * TMW) * ldc + (nb + wn * TNW) / 2 + c * 8;
        const int clim = (ncols - nb - wn * TNW) / 2;
        // G and U rounded and packed first: half the registers, and every output forms from the rounded values
        uint32_t pk[FM][FN][2];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              pk[i][j][h] = pack2<T>(acc[i][j][2 * h], acc[i][j][2 * h + 1]);
              asm volatile("" : "+v"(pk[i][j][h]));  // the packed value, not the accumulators, is what stays live
            }
        auto emit = [&](auto out_c, u16* dst) {
          constexpr int out = decltype(out_c)::value;
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int p = 0; p < FN / 2; ++p) {
              const uint32_t(&g)[2] = pk[i][2 * p];
              const uint32_t(&u)[2] = pk[i][2 * p + 1];
              uint32_t o[2];
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const float g0 = to_f32<T>((u16)(g[h] & 0xffffu)), g1 = to_f32<T>((u16)(g[h] >> 16));
                const float u0 = to_f32<T>((u16)(u[h] & 0xffffu)), u1 = to_f32<T>((u16)(u[h] >> 16));
                o[h] = out == 0 ? g[h] : out == 1 ? u[h] : pack2<T>(g0 * q3_sigmoid(g0) * u0, g1 * q3_sigmoid(g1) * u1);
              }
              stage_out(i, p, o[0], o[1]);
            }
          lds_wait();
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int q = 0; q < (TMW + RPI - 1) / RPI; ++q) {
            const int r = q * RPI + lane / CH;
            if (r < min(rlim, TMW) && c * 8 < clim) *reinterpret_cast<i32x4*>(dst + (int64_t)r * ldc) = row_chunk(r);
          }
          lds_wait();
          __builtin_amdgcn_wave_barrier();
        };
        if (ar.g) {
          emit(std::integral_constant<int, 0>{}, ar.g + o0);
          emit(std::integral_constant<int, 1>{}, ar.u + o0);
        }
        emit(std::integral_constant<int, 2>{}, C + o0);
        return;
      } else {
        const int clim = ncols - nb - wn * TNW;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            stage_out(i, j, pack2<T>(acc[i][j][0], acc[i][j][1]), pack2<T>(acc[i][j][2], acc[i][j][3]));
        const int64_t r0 = (int64_t)(ma + wm * TMW), c0 = nb + wn * TNW + c * 8;
        lds_wait();
        __builtin_amdgcn_wave_barrier();
        // batches of up to 4 row passes: the batch's residual (or g / u) rows are all in flight before their use
        constexpr int NP = TMW / RPI, BP = NP % 4 == 0 ? 4 : NP % 3 == 0 ? 3 : NP < 4 ? NP : 1;
        static_assert(NP % BP == 0, "row passes");
#pragma unroll
        for (int q0 = 0; q0 < NP; q0 += BP) {
          i32x4 x0[BP], x1[BP];
          if (EPI == 5 || ar.res) {
#pragma unroll
            for (int q = 0; q < BP; ++q) {
              const int r = (q0 + q) * RPI + lane / CH;
              if (r >= rlim || c * 8 >= clim) continue;
              if constexpr (EPI == 5) {
                x0[q] = *reinterpret_cast<const i32x4*>(ar.gin + (r0 + r) * ar.ldgu + c0);
                x1[q] = *reinterpret_cast<const i32x4*>(ar.uin + (r0 + r) * ar.ldgu + c0);
              } else {
                x0[q] = *reinterpret_cast<const i32x4*>(ar.res + (r0 + r) * ar.ldres + c0);
              }
            }
          }
#pragma unroll
          for (int q = 0; q < BP; ++q) {
            const int r = (q0 + q) * RPI + lane / CH;
            if (r >= rlim || c * 8 >= clim) continue;
            i32x4 v = row_chunk(r);
            if constexpr (EPI == 5) {
              const Vec<T> df = unpack_vec<T>(v), gf = unpack_vec<T>(x0[q]), uf = unpack_vec<T>(x1[q]);
              Vec<T> og, ou;
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const float sg = q3_sigmoid(gf.v[e]);
                og.v[e] = df.v[e] * uf.v[e] * sg * (1.f + gf.v[e] * (1.f - sg));
                ou.v[e] = df.v[e] * gf.v[e] * sg;
              }
              store_vec<T>(reinterpret_cast<u16*>(ar.c[0]) + (r0 + r) * ldc + c0, og);
              store_vec<T>(reinterpret_cast<u16*>(ar.c[1]) + (r0 + r) * ldc + c0, ou);
            } else {
              if (ar.res) {  // C = res + round(product), rounded again: the GEMM followed by the add kernel
                const Vec<T> p = unpack_vec<T>(v), b = unpack_vec<T>(x0[q]);
#pragma unroll
                for (int w = 0; w < 4; ++w)
                  v[w] = (int)pack2<T>(p.v[2 * w] + b.v[2 * w], p.v[2 * w + 1] + b.v[2 * w + 1]);
              }
              *reinterpret_cast<i32x4*>(C + (r0 + r) * ldc + c0) = v;
            }
          }
        }
        return;
      }
    }
  }
  if constexpr (EPI == 0) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = ma + wm * TMW + i * 16 + j16;
      if (row >= mrows) continue;
      u16* crow = C + (int64_t)row * ldc;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = nb + wn * TNW + j * 16 + 4 * quarter;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (col + v < ncols) {
            float x = to_f32<T>(from_f32<T>(acc[i][j][v]));
            if (ar.res) x += to_f32<T>(ar.res[(int64_t)row * ar.ldres + col + v]);
            crow[col + v] = from_f32<T>(x);
          }
      }
    }
  }
}

template <typename T, int BM, int BN, int WM, int WN, int ST, bool AT, bool BT, int EPI, bool KP = false>
int launch_tile(const Args& a, hipStream_t s) {
  const int64_t tiles = (int64_t)a.tms * a.tns * a.splits;
  gemm_tile_kernel<T, BM, BN, WM, WN, ST, AT, BT, EPI, KP><<<(unsigned)tiles, WM * WN * 64, 0, s>>>(a);
  return (int)hipGetLastError();
}

}  // namespace q3gemm
