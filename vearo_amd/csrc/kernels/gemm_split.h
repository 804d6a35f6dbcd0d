// gemm_split.h -- f32 matrix multiply for large dense products on the bf16
// matrix cores: every operand value is split into three bf16 parts as it is
// staged, and six part products per pair carry the f32 product (split3.h).
//
// Semantics, work split and epilogue of gemm_big.h, the same product on the f32
// instruction: C = alpha A B (+ E) (+ C), each operand k-contiguous or
// row-contiguous, one 512-thread workgroup per CU walking a list of (C tile, k
// range) segments as one continuous stream of k tiles, whole-tile rounds and a
// last round that is split along K over all workgroups or left whole
// (a.whole_tail), a fix-up adding the pieces in k order. Here any K runs in
// whole: the last k tile is masked in LDS. A tile of a round left whole may be summed
// in several chains of k tiles (a.whole_tail of them), each added to C by the thread
// that stored the ones before: the host asks for it where one chain would round
// more than the pieces of a split round (gemm_split_plan).
//
// What bounds it: the chip's power. On MI355X the matrix cores hold 2.4 GHz on
// zeros (lm_head dx [16384, 50272] x [50272, 768]: 3.86 ms, 328 TFLOP/s of f32
// products) and ~1.6 GHz on random data (5.63 ms, 225; matrix cores busy 0.77 of
// the cycles), as a large bf16 library product does here (1340 TFLOP/s, a sixth
// of which is 223). The f32 instruction's kernel takes 8.65 ms; lm_head forward
// 8.88 -> 5.65 ms, [16384, 768] x [768, 3072] 556 -> 343 us, x [768, 768] 155 -> 95,
// the weight gradient [3072 x 16384] x [16384 x 768] 594 -> 375. Three other
// schedules of the k step (the compiler's own, grouped by instruction kind, 16
// more products before the barrier) ran within 2 % of this one on random data
// and up to 8 % slower on zeros; part products ordered to share an operand with
// the one before, or LDS without the ~8 conflict cycles of the k-contiguous
// writes, changed nothing.
//
// Tile: 256 x BN (256, or 192 where that fits N and the chip better: vh_gemm's
// plan), 8 waves, two per SIMD, of 64 x BN / 2 as 2 x BN / 64 matrix-core tiles. K
// advances in tiles of 16 through two LDS stages of 49 KB: the k step on tile p
// splits tile p + 1 (in registers since the previous step) into the free stage and
// reloads the registers with tile p + 2. Splitting costs 5.5 vector instructions
// per value, once per workgroup (a wave that split its fragments after reading
// them would do 3 times as many), ~2 per matrix instruction, in their shadow.
//
// Signs. The matrix core adds a group of eight products and the accumulator with
// 8 bits below the accumulator's last and drops what is below those by rounding
// down (measured), so sums drift towards minus infinity: by up to ~1e-8 of the
// accumulator per 16 k where the small part products reach below those bits. Left
// alone that bias survives sums over outputs (the final layer norm's bias gradient
// of the GPT step was 6.5e-6 off, 0.98 of it common to all elements, against 6.7e-7
// on the f32 instruction). So A enters negated in every other run of GS_FLIP k
// tiles and every other group of 32 rows, B in every other 32 columns, and the
// accumulators are negated at each run's start: the drift changes direction and
// cancels, along K and over rows and columns. (The factor that split3.h puts on
// each value carries the sign; 1/8 negation per accumulator and k tile.) What stays is
// per row and column: with one-signed operands the small part products of a row's
// (column's) l with the other operand's h round away under the sum alike for all its
// elements, so a row's or column's mean is 0.8 u of it off at K = 768 and 3072, 0.5 u
// at 16384 (f32 instruction: 0.1, 0.2; u = 2^-24), while the elements themselves are
// 2.8e-7, 4.7e-7 and 1.2e-6 off against 3.7e-7, 7.4e-7 and 2.0e-6.
#pragma once
#include <type_traits>

#include "common.h"
#include "gemm_big.h"
#include "split3.h"

#define GS_TK VH_GEMMS_TK
#define GS_FLIP 8  // k tiles per run of one sign, a power of two

// LDS of one operand's 256 x 16 k tile: its three parts, each as two k halves
// of [row] 16-byte pieces (8 k of a row, the matrix cores' fragment).
#define GS_HALF (256 * 4 + 16)   // dwords per k half
#define GS_PART (2 * GS_HALF)    // dwords per part
#define GS_STAGE (3 * GS_PART)   // dwords per operand and stage

// The work split shared by the kernel and the fix-up: G workgroups, `full`
// whole-tile rounds, then W = rem * nk k tiles split evenly (the host keeps
// tile and k tile counts, and W, below 2^31). With a.whole_tail the rem tiles
// of the last round are not split: rem of the workgroups take one each.
struct GsSplit {
  int tiles, nk, full, rem, W, G;
  VH_DEV GsSplit(const GemmArgs& a, int G_) : G(G_) {
    tiles = a.tiles_m * a.tiles_n * (int)a.nbat;  // tiles of all batches (the host keeps it < 2^31)
    nk = (int)((a.K + GS_TK - 1) / GS_TK);
    full = tiles / G;
    rem = tiles - full * G;
    W = a.whole_tail ? 0 : rem * nk;
  }
  VH_DEV int begin(int g) const { return (int)((int64_t)W * g / G); }
  VH_DEV int end(int g) const { return (int)((int64_t)W * (g + 1) / G); }
};

template <bool A_KC, bool B_KC, int BN>
VH_DEV void gemm_split_impl(const GemmArgs& a) {
  static_assert(BN == 256 || BN == 192, "tile width");
  // A wave's block: 64 x BN / 2 as 2 x NB matrix-core tiles of 32 x 32.
  constexpr int WM = 2, NB = BN / 64, WR = 64, WC = BN / 2;
  __shared__ __attribute__((aligned(1024))) uint32_t L[2][2][GS_STAGE];  // [stage][A, B]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1, li = lane & 31, h = lane >> 5;
  const int G = (int)gridDim.x, g = (int)blockIdx.x;
  const GsSplit sp(a, G);

  // This workgroup's segments: `full` whole tiles, then the pieces of its
  // stream-K run [sb, se) cut at tile boundaries.
  if (sp.nk == 0) return;
  const int sb = sp.begin(g), se = sp.end(g);
  const int t0 = sb / sp.nk;
  const int npieces = se > sb ? (se - 1) / sp.nk - t0 + 1 : 0;
  // XCD-major position in a round: XCD x (= g % 8, the hardware's round-robin)
  // takes G / 8 consecutive tiles, or its eighth of an unsplit last round.
  const int x = g % 8, local = x * (G / 8) + g / 8;
  const int xlo = sp.rem * x / 8, xn = sp.rem * (x + 1) / 8 - xlo;
  const int nch = a.whole_tail > 1 ? a.whole_tail : 1;  // chains per whole tile
  const int ndp = (sp.full + (a.whole_tail && g / 8 < xn ? 1 : 0)) * nch;  // whole-tile segments
  const int nseg = ndp + npieces;
  if (nseg == 0) return;
  auto seg_of = [&](int j) {
    GbSeg s;
    int u, kt0 = 0, kt1 = sp.nk;
    s.slot = -1;
    if (j < ndp) {
      const int t = j / nch, c = j - t * nch;
      u = t * G + (t < sp.full ? local : xlo + g / 8);
      kt0 = sp.nk * c / nch;  // (the host keeps nk * nch below 2^31)
      kt1 = sp.nk * (c + 1) / nch;
    } else {
      const int p = j - ndp, t = t0 + p;  // (never with whole_tail)
      u = sp.full * G + t;
      const int lo = t * sp.nk;
      kt0 = (sb > lo ? sb : lo) - lo;
      kt1 = (se < lo + sp.nk ? se : lo + sp.nk) - lo;
      if (kt0 != 0 || kt1 != sp.nk) s.slot = p == 0 ? 0 : 1;
    }
    int tm, tn;
    gb_locate(a, u, tm, tn, s);
    s.m0 = tm * GB_TM;
    s.n0 = tn * BN;
    s.kt0 = kt0;
    s.kt1 = kt1;
    return s;
  };

  // Staging: each thread brings eight consecutive k of one row of each
  // operand's 256 x 16 k tile, as two 128-bit loads.
  //   k-contiguous: thread t takes k half t & 1 of row t / 2 (two threads
  //     cover a row's 64 bytes); its LDS piece is the row's.
  //   row-contiguous: lane 16 q + c of wave w loads rows 4 c .. 4 c + 3 of 64-row
  //     block w & 3 at k = 2 q and 2 q + 1 of k half w >> 2 (256 contiguous bytes
  //     per k); a 4 x 4 transpose across the lanes' q then leaves lane (q, c)
  //     with all eight k of row 4 c + q. Its piece goes to 16 q + (c + 4 q) % 16 of
  //     the block: the writes of 16 lanes, and the reads of 16 consecutive
  //     rows, each touch 16 different 16-byte bank groups.
  const int q4 = lane >> 4, c4 = lane & 15;
  const int rt = 64 * (w & 3) + 16 * q4 + ((c4 + 4 * q4) & 15);  // row-contiguous: LDS piece
  const int ka = A_KC ? tid & 1 : w >> 2, kb = B_KC ? tid & 1 : w >> 2;
  const uint32_t lda4 = (uint32_t)a.lda * 4u, ldb4 = (uint32_t)a.ldb * 4u;
  const uint32_t okc = (64 * (w & 3) + 4 * c4) * 4u;
  const uint32_t oa = A_KC ? (uint32_t)(tid >> 1) * lda4 + ka * 32u : (uint32_t)(8 * ka + 2 * q4) * lda4 + okc;
  // (A narrower tile leaves the waves of B's rows from BN on without work: their
  // offset is past any record, so they load zeros from nowhere.)
  const bool bidle = B_KC ? w >= BN / 32 : (w & 3) >= BN / 64;
  const uint32_t ob = bidle  ? 0xFFFFFF00u
                      : B_KC ? (uint32_t)(tid >> 1) * ldb4 + kb * 32u
                             : (uint32_t)(8 * kb + 2 * q4) * ldb4 + okc;
  const uint32_t oa2 = A_KC ? 16u : lda4, ob2 = B_KC || bidle ? 16u : ldb4;  // second load
  const int wa = ka * GS_HALF + (A_KC ? tid >> 1 : rt) * 4, wb = kb * GS_HALF + (B_KC ? tid >> 1 : rt) * 4;
  vh_f4 ga[2], gb[2];
  // Factors (see above): S3_SCALE, negative in every other run of GS_FLIP k tiles
  // and every other group of 32 rows of A, and every other 32 columns of B.
  auto run_sign = [](int kt) { return kt & GS_FLIP ? -1.0f : 1.0f; };
  auto row8 = [](auto kc, const vh_f4 (&v)[2], float (&x)[8]) {
    if constexpr (decltype(kc)::value) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = v[e >> 2][e & 3];
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const vh_u4 u = __builtin_bit_cast(vh_u4, v[e]);
        uint32_t t[4] = {u[0], u[1], u[2], u[3]};
        s3_transpose4(t);
#pragma unroll
        for (int j = 0; j < 4; ++j) x[2 * j + e] = __builtin_bit_cast(float, t[j]);
      }
    }
  };
  // The staged k tile's pieces: pair i of a row's eight k is split at a time
  // (see kstep); the parts collect in sp, then go to stage st.
  vh_u4 sp3[3];
  float x8[8];
  auto scale = [&](float f) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x8[e] *= f;
  };
  auto split_pair = [&](int i) {
    uint32_t h0, m0, l0;
    s3_split2(x8[2 * i], x8[2 * i + 1], h0, m0, l0);
    sp3[0][i] = h0;
    sp3[1][i] = m0;
    sp3[2][i] = l0;
  };
  auto write_a = [&](int st) {
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<vh_u4*>(&L[st][0][t * GS_PART + wa]) = sp3[t];
  };
  auto write_b = [&](int st) {
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<vh_u4*>(&L[st][1][t * GS_PART + wb]) = sp3[t];
  };
  const float fsa = (A_KC ? tid >> 6 : c4 >> 3) & 1 ? -S3_SCALE : S3_SCALE;
  const float fsb = (B_KC ? tid >> 6 : c4 >> 3) & 1 ? -S3_SCALE : S3_SCALE;
  const std::integral_constant<bool, A_KC> akc{};
  const std::integral_constant<bool, B_KC> bkc{};
  // A k tile with only kv of its 16 k inside K: what the loads returned past K
  // (another row's values, or zeros past the operand) becomes zero in both
  // operands. Each thread masks its own pieces in LDS, before the barrier.
  auto mask_tail = [&](int st, int kv) {
    auto mask = [&](vh_u4* p, int k0) {
      vh_u4 v = *p;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] &= k0 + 2 * i + 1 < kv ? 0xFFFFFFFFu : k0 + 2 * i < kv ? 0xFFFFu : 0u;
      *p = v;
    };
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      mask(reinterpret_cast<vh_u4*>(&L[st][0][t * GS_PART + wa]), 8 * ka);
      mask(reinterpret_cast<vh_u4*>(&L[st][1][t * GS_PART + wb]), 8 * kb);
    }
  };
  // Barrier for LDS only: the staging loads in flight are not waited for.
  auto lds_barrier = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // The load cursor walks the same k tile stream two tiles ahead of the
  // products: segment lj, `left` k tiles of it still to come after this one,
  // the tile's origin in each operand and the bytes from there to the
  // operand's last element, stepped from one k tile to the next (a record count
  // of none past the end of the stream: reads give 0).
  int lj = 0, left = 0, kleft = 0, lkt = 0;
  const char *pa = nullptr, *pb = nullptr;
  int64_t na = 0, nb = 0, da = A_KC ? GS_TK * 4 : GS_TK * 4 * a.lda, db = B_KC ? GS_TK * 4 : GS_TK * 4 * a.ldb;
  auto seek = [&](const GbSeg& sg) {
    const int64_t k0 = (int64_t)sg.kt0 * GS_TK, m0 = sg.m0, n0 = sg.n0;
    pa = reinterpret_cast<const char*>(a.A + sg.ao + (A_KC ? m0 * a.lda + k0 : k0 * a.lda + m0));
    pb = reinterpret_cast<const char*>(a.B + sg.bo + (B_KC ? n0 * a.ldb + k0 : k0 * a.ldb + n0));
    na = (A_KC ? (a.M - 1 - m0) * a.lda + a.K - k0 : (a.K - 1 - k0) * a.lda + a.M - m0) * 4;
    nb = (B_KC ? (a.N - 1 - n0) * a.ldb + a.K - k0 : (a.K - 1 - k0) * a.ldb + a.N - n0) * 4;
    left = sg.kt1 - sg.kt0 - 1;
    lkt = sg.kt0;
    kleft = (int)(a.K - k0);
  };
  auto advance = [&]() {
    if (left > 0) {
      --left;
      ++lkt;
      kleft -= GS_TK;
      pa += da;
      pb += db;
      na -= da;
      nb -= db;
    } else if (++lj < nseg) {
      seek(seg_of(lj));
    } else {
      kleft = GS_TK;
      na = nb = 0;
      lj = nseg;
    }
  };
  // (The offsets are opaque at each use: the second load's is then formed there,
  // as the instruction's immediate or one addition, instead of held in a register.)
  auto load2 = [](const char* p, int64_t n, uint32_t o, uint32_t o2, vh_f4 (&v)[2]) {
    const auto r = gm_rsrc(reinterpret_cast<const float*>(p), n);
    asm volatile("" : "+v"(o));
    v[0] = gm_bload(r, o);
    v[1] = gm_bload(r, o + o2);
  };
  auto load_a = [&]() { load2(pa, na, oa, oa2, ga); };
  auto load_b = [&]() { load2(pb, nb, ob, ob2, gb); };
  GbSeg cur = seg_of(0);
  seek(cur);
  load_a();
  load_b();
  row8(akc, ga, x8);
  scale(fsa * run_sign(lkt));
  for (int i = 0; i < 4; ++i) split_pair(i);
  write_a(0);
  row8(bkc, gb, x8);
  scale(fsb);
  for (int i = 0; i < 4; ++i) split_pair(i);
  write_b(0);
  if (kleft < GS_TK) mask_tail(0, kleft);
  advance();
  int kv = kleft;  // k inside K of the tile in the staging registers, and its sign
  float sgn = run_sign(lkt);
  load_a();
  load_b();
  lds_barrier();
  vh_f32x16 acc[WM][NB];

  // Fragments: lane (li, h) of a 32-row group holds k = 8 h .. 8 h + 7 of row li.
  // Row 32 i + li of a 64-row block sits at its own piece (k-contiguous) or, for
  // a row-contiguous operand, where the staging put it (odd i: the same piece ^ 8).
  const int lt = 16 * (li & 3) + (((li >> 2) + 4 * (li & 3)) & 15);
  const int fa0 = h * GS_HALF + (wm * WR + (A_KC ? li : lt)) * 4, fa1 = A_KC ? fa0 + 128 : fa0 + 4 * ((lt ^ 8) - lt);
  // B's 32-row group jj of wave column wn is group wn BN / 64 + jj: groups jj = 0, 2
  // share a parity, and so a base, and jj = 1, 3 the other.
  const int bg = wn * NB;
  auto b_base = [&](int grp) {
    return h * GS_HALF + (B_KC ? 32 * grp + li : 64 * (grp >> 1) + (grp & 1 ? lt ^ 8 : lt)) * 4;
  };
  const int fb0 = b_base(bg), fb1 = b_base(bg + 1);
  constexpr int SETS = NB == 3 ? 3 : 2;  // B fragment sets: the last group's is not the first's
  vh_u4 fa[WM][3], fb[SETS][3];
  auto read_a1 = [&](int st, int i, int t) {
    fa[i][t] = *reinterpret_cast<const vh_u4*>(&L[st][0][t * GS_PART + (i ? fa1 : fa0)]);
  };
  auto read_a = [&](int st, int i) {
#pragma unroll
    for (int t = 0; t < 3; ++t) read_a1(st, i, t);
  };
  auto read_b = [&](int st, int jj) {
#pragma unroll
    for (int t = 0; t < 3; ++t) fb[jj % SETS][t] = *reinterpret_cast<const vh_u4*>(&L[st][1][t * GS_PART + (jj & 1 ? fb1 : fb0) + 256 * (jj >> 1)]);
  };
  // Part products t0 .. t0 + n - 1 of tile (i, jj).
  auto products = [&](int i, int jj, int t0, int n) {
#pragma unroll
    for (int t = t0; t < t0 + n; ++t) acc[i][jj] = s3_mfma(fa[i][S3_PA(t)], fb[jj % SETS][S3_PB(t)], acc[i][jj]);
  };
  read_a(0, 0);
  read_b(0, 0);
  read_a(0, 1);

  // One k step on stage st, laid out in chunks that the compiler's scheduler
  // keeps apart: a quarter of an operand's split (11 vector instructions) per
  // three products, so that neither unit waits for a run of the other's; each
  // operand's loads go out as soon as its registers are free, three quarters of
  // a step before they are needed.
  auto chunk = []() { __builtin_amdgcn_sched_barrier(0); };
  auto kstep = [&](int st) {
    read_b(st, 1);
    row8(akc, ga, x8);
    scale(fsa * sgn);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      products(c >> 1, 0, 3 * (c & 1), 3);
      split_pair(c);
      chunk();
    }
    write_a(st ^ 1);
    load_a();
    read_b(st, 2);
    row8(bkc, gb, x8);
    scale(fsb);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      products(c >> 1, 1, 3 * (c & 1), 3);
      split_pair(c);
      chunk();
    }
    write_b(st ^ 1);
    load_b();
    if constexpr (NB == 4) {
      read_b(st, 3);
      products(0, 2, 0, 6);
      products(1, 2, 0, 6);
    }
    if (kv < GS_TK) mask_tail(st ^ 1, kv);
    lds_barrier();
    chunk();
    // The next step's first fragments, each A part as its last product goes out.
    read_b(st ^ 1, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      products(i, NB - 1, 0, 1);
      chunk();
      read_a1(st ^ 1, i, 2);
      products(i, NB - 1, 1, 3);
      chunk();
      read_a1(st ^ 1, i, 1);
      products(i, NB - 1, 4, 2);
      chunk();
      read_a1(st ^ 1, i, 0);
    }
  };
  int s = 0;
  // What redo and epilogue read of the arguments they load again from the kernel's
  // argument segment, behind a barrier to the compiler: held in scalar registers across
  // the k loop, they would push its own into vector lanes.
  auto args = []() {
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return (const GemmArgs*)p;
  };
  // The infinities and NaN of a wave's block again, a 32 x 32 tile at a time on the f32
  // instruction straight from memory (see split3.h). [16384, 768] x [768, 3072] full of
  // NaN takes 1.36 ms (operands k-contiguous) or 1.87 (row-contiguous) against 0.34 of
  // numbers, with one infinity 0.45 or 0.54. Two or more tiles at a time would share
  // their loads (1.13 and 1.27), but take registers from the usual path (0.34 -> 0.35).
  // A row past M (column past N) reads the last one's: none of its outputs is replaced.
  auto redo = [&]() {
    const GemmArgs& a = *args();
    const int64_t k1 = (int64_t)cur.kt1 * GS_TK < a.K ? (int64_t)cur.kt1 * GS_TK : a.K;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int jj = 0; jj < NB; ++jj) {
        int l = li;
        asm volatile("" : "+v"(l));  // (addresses formed here, as below)
        const int64_t m0 = cur.m0 + wm * WR + 32 * i, m = m0 + l, n = cur.n0 + wn * WC + 32 * jj + l;
        const uint32_t bad = s3_nonfinite_regs(acc[i][jj], a.M - m0 - 4 * h, a.N - n);
        if (__builtin_amdgcn_ballot_w64(bad != 0) == 0) continue;
        // Lane half h takes k + 4 h .. k + 4 h + 3 of every eight k, one load where they lie
        // together.
        const int64_t k0 = (int64_t)cur.kt0 * GS_TK + 4 * h;
        const int64_t mc = m < a.M ? m : a.M - 1, nc = n < a.N ? n : a.N - 1;
        const float* pa = a.A + cur.ao + (A_KC ? mc * a.lda + k0 : k0 * a.lda + mc);
        const float* pb = a.B + cur.bo + (B_KC ? nc * a.ldb + k0 : k0 * a.ldb + nc);
        auto load = [&](auto kc, const float* p, int64_t ld, int left, float (&v)[4]) {
          if (decltype(kc)::value && left >= 8) {
            const s3_f4u q = *reinterpret_cast<const s3_f4u*>(p);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = q[u];
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = 4 * h + u < left ? p[decltype(kc)::value ? u : u * ld] : 0.0f;
          }
        };
        vh_f32x16 t{};
#pragma nounroll
        for (int left = (int)(k1 - (int64_t)cur.kt0 * GS_TK); left > 0; left -= 8) {
          float x[4], y[4];
          load(akc, pa, a.lda, left, x);
          load(bkc, pb, a.ldb, left, y);
#pragma unroll
          for (int u = 0; u < 4; ++u) t = __builtin_amdgcn_mfma_f32_32x32x2f32(x[u], y[u], t, 0, 0, 0);
          pa += A_KC ? 8 : 8 * a.lda;
          pb += B_KC ? 8 : 8 * a.ldb;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][jj][r] = bad >> r & 1 ? t[r] : acc[i][jj][r];
      }
  };
  // The current segment's epilogue straight from the accumulators: register
  // r of a 32 x 32 tile holds row 8 (r / 4) + 4 h + r % 4, column li. A
  // partial piece goes raw to its workspace slot, a whole tile to C as
  // alpha v (+ E) (+ C) inside M x N. The row stride and this lane's row and
  // column are opaque here, so that the compiler forms the per-element
  // offsets where they are used instead of keeping them in registers across
  // the whole segment loop.
  auto epilogue = [&]() {
    const GemmArgs& a = *args();
    const bool raw = cur.slot >= 0;
    int64_t ldo = raw ? BN : a.ldc;
    int lrow = wm * WR + 4 * h, lcol = wn * (BN / 2) + li;
    asm volatile("" : "+s"(ldo), "+v"(lrow), "+v"(lcol));
    const int64_t slot_elems = (int64_t)GB_TM * BN;
    if (raw) {
      float* base = a.ws + ((int64_t)g * GB_SLOTS + cur.slot) * slot_elems + lrow * BN + lcol;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float* row = base + (32 * i + 8 * (r >> 2) + (r & 3)) * BN;
#pragma unroll
          for (int jj = 0; jj < NB; ++jj) row[32 * jj] = acc[i][jj][r];
        }
      return;
    }
    using T = std::true_type;
    using F = std::false_type;
    const bool inner = cur.m0 + GB_TM <= a.M && cur.n0 + BN <= a.N;
    float* const Cb = a.C + cur.co;
    const bool more = cur.kt0 > 0;  // a further chain: C holds the ones before, E and the old C among them
    const float* const Eb = a.E && !more ? a.E + cur.eo : nullptr;
    const bool accumulate = a.accumulate || more;
    if (inner && !Eb && !accumulate) {
      float* base = Cb + (cur.m0 + lrow) * ldo + cur.n0 + lcol;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float* row = base + (32 * i + 8 * (r >> 2) + (r & 3)) * ldo;
#pragma unroll
          for (int jj = 0; jj < NB; ++jj) row[32 * jj] = acc[i][jj][r] * a.alpha;
        }
      return;
    }
    if (inner && (!Eb || a.sem == 0)) {
      // Whole tile inside C with at most a per-column addend (a bias, E
      // stride 0 along m, read once per column): v = alpha acc (+ bias)
      // (+ old C), in gm_finish's order, no bounds tests. The stores may
      // alias the old-C reads as far as the compiler knows, so it keeps
      // each read behind the stores before it: the reads go out 8 rows x
      // NB columns at a time, ahead of their stores, so a wave waits on
      // memory 2 WM times, not once per element.
      float* base = Cb + (cur.m0 + lrow) * ldo + cur.n0 + lcol;
      float eb[NB];
#pragma unroll
      for (int jj = 0; jj < NB; ++jj) eb[jj] = Eb ? Eb[(cur.n0 + lcol + 32 * jj) * a.sen] : 0.0f;
      auto tile = [&](auto has_bias, auto acc_c) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int r0 = 0; r0 < 16; r0 += 8) {
            float old[8][NB];
            if constexpr (decltype(acc_c)::value) {
#pragma unroll
              for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int jj = 0; jj < NB; ++jj)
                  old[r][jj] = base[(32 * i + 8 * ((r0 + r) >> 2) + ((r0 + r) & 3)) * ldo + 32 * jj];
            }
#pragma unroll
            for (int r = 0; r < 8; ++r) {
              float* row = base + (32 * i + 8 * ((r0 + r) >> 2) + ((r0 + r) & 3)) * ldo;
#pragma unroll
              for (int jj = 0; jj < NB; ++jj) {
                float v = acc[i][jj][r0 + r] * a.alpha;
                if constexpr (decltype(has_bias)::value) v = v + eb[jj];
                if constexpr (decltype(acc_c)::value) v = old[r][jj] + v;
                row[32 * jj] = v;
              }
            }
          }
      };
      if (Eb) {
        if (accumulate) tile(T{}, T{}); else tile(T{}, F{});
      } else {
        tile(F{}, T{});  // accumulate (the plain store returned above)
      }
      return;
    }
    if (inner) {
      // Whole tile inside C with a full addend E[m, n]: v = alpha acc + E
      // (+ old C), in gm_finish's order, without bounds tests.
      float* base = Cb + (cur.m0 + lrow) * ldo + cur.n0 + lcol;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int rl = 32 * i + 8 * (r >> 2) + (r & 3);
          float* row = base + rl * ldo;
#pragma unroll
          for (int jj = 0; jj < NB; ++jj) {
            float v = acc[i][jj][r] * a.alpha;
            v = v + Eb[(cur.m0 + lrow + rl) * a.sem + (cur.n0 + lcol + 32 * jj) * a.sen];
            if (accumulate) v = row[32 * jj] + v;
            row[32 * jj] = v;
          }
        }
      return;
    }
    // A tile at an edge of C: rows below mlim and columns below nlim of this lane's. The
    // reads of old C again go out 8 rows x NB columns at a time, and are waited for once:
    // under per-element tests the compiler would wait for everything at each element.
    const int64_t mr = a.M - cur.m0 - lrow, nr = a.N - cur.n0 - lcol;
    int mlim = mr < GB_TM ? (int)mr : GB_TM, nlim = nr < BN ? (int)nr : BN;
    float* base = Cb + (cur.m0 + lrow) * ldo + cur.n0 + lcol;
    if (Eb && a.sem != 0) {  // a full addend
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          asm volatile("" : "+v"(mlim), "+v"(nlim));  // (tests and offsets formed here, as above)
          const int rl = 32 * i + 8 * (r >> 2) + (r & 3);
#pragma unroll
          for (int jj = 0; jj < NB; ++jj)
            if (rl < mlim && 32 * jj < nlim) {
              float v = acc[i][jj][r] * a.alpha;
              v = v + Eb[(cur.m0 + lrow + rl) * a.sem + (cur.n0 + lcol + 32 * jj) * a.sen];
              if (accumulate) v = base[rl * ldo + 32 * jj] + v;
              base[rl * ldo + 32 * jj] = v;
            }
        }
      return;
    }
    float eb[NB];
#pragma unroll
    for (int jj = 0; jj < NB; ++jj) eb[jj] = Eb && 32 * jj < nlim ? Eb[(cur.n0 + lcol + 32 * jj) * a.sen] : 0.0f;
    auto edge = [&](auto has_bias, auto acc_c) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += 8) {
          asm volatile("" : "+v"(mlim), "+v"(nlim));
          float old[8][NB];
          if constexpr (decltype(acc_c)::value) {
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
              for (int jj = 0; jj < NB; ++jj) {
                const int rl = 32 * i + 8 * ((r0 + r) >> 2) + ((r0 + r) & 3);
                old[r][jj] = rl < mlim && 32 * jj < nlim ? base[rl * ldo + 32 * jj] : 0.0f;
              }
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
          }
#pragma unroll
          for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int jj = 0; jj < NB; ++jj) {
              const int rl = 32 * i + 8 * ((r0 + r) >> 2) + ((r0 + r) & 3);
              float v = acc[i][jj][r0 + r] * a.alpha;  // (gm_finish's order)
              if constexpr (decltype(has_bias)::value) v = v + eb[jj];
              if constexpr (decltype(acc_c)::value) v = old[r][jj] + v;
              if (rl < mlim && 32 * jj < nlim) base[rl * ldo + 32 * jj] = v;
            }
        }
    };
    if (Eb) {
      if (accumulate) edge(T{}, T{}); else edge(T{}, F{});
    } else {
      if (accumulate) edge(F{}, T{}); else edge(F{}, F{});
    }
  };
  // Segments in order; per segment, one k step per k tile on alternating
  // stages (the staged tile -- the next in the stream -- goes to LDS and the
  // one after it is loaded), then the epilogue.
  for (int j = 0;;) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int jj = 0; jj < NB; ++jj) acc[i][jj] = vh_f32x16{};
    // Nothing but the staged loads is in flight in the loop, and those have had
    // the epilogue to arrive: waiting here keeps the compiler from fencing
    // every k step against the epilogue's memory operations.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    for (int kt = cur.kt0; kt < cur.kt1; ++kt) {
      if ((kt & (GS_FLIP - 1)) == 0) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int jj = 0; jj < NB; ++jj) acc[i][jj] = -acc[i][jj];
      }
      advance();
      kstep(s);
      kv = kleft;
      sgn = run_sign(lkt);
      s ^= 1;
    }
    // Back to the products' own scale and sign (+ 0: a sum of zeros is +0).
    const float un = ((cur.kt1 - 1) & GS_FLIP ? 1 : 0) ^ (bg & 1) ? -S3_UNSCALE : S3_UNSCALE;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int jj = 0; jj < NB; ++jj)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][jj][r] = __builtin_fmaf(acc[i][jj][r], (i ^ jj) & 1 ? -un : un, 0.0f);
    if (s3_nonfinite(acc)) redo();
    epilogue();
    if (++j == nseg) break;
    cur = seg_of(j);
  }
}
