// gemm.h -- f32 matrix multiply on the gfx950 matrix cores, each operand value split
// in three bf16 parts (split3.h).
//
// Semantics: vearo-backend-cpu matmul (crates/vearo-backend-cpu/src/lib.rs:266-417),
// C[m, n] = sum_k A[m, k] * B[k, n] in f32 (the matrix core accumulates in f32;
// the grouping of the k sum differs from the CPU's sequential mul_add chain,
// which is within f32 rounding). The epilogue applies, in this order,
//   v = acc * alpha;  v = v + E[m, n] (optional addend);  v = C[m, n] + v (optional)
// which are exactly the separate ops the reference runs after a matmul:
// `* scale` and `+ mask` in attention (cpu:2431-2449), `+ bias` in Linear
// (nn:120-128), and gradient accumulation `existing.add(g)` (autograd:733-742).
//
// Tiling: GemmTile below, 128 x 128 or 64 x 64 C tiles; K in tiles of 32.
// A operand layouts: k-contiguous (A[m, k] at m*lda + k) or m-contiguous
// (A[m, k] at k*lda + m, a transposed view); the same for B.
//
// Causal modes for attention's score blocks (the masked part is exactly 0 or
// never read, so skipping it changes no result):
//   1: skip tiles entirely above the diagonal (n > m for all elements);
//   2: only k <= m contributes (P V and dS K: row m's weights are 0 past m);
//   3: only k >= m contributes (P^T dO and dS^T Q).
#pragma once
#include "common.h"
#include "split3.h"

#define GM_TM VH_GEMM_TILE_M
#define GM_TK 32
#define GM_GROUP 8         // tile rows per group in the launch order (L2 reuse of B)

template <bool B>
struct GmFlag {
  static constexpr bool value = B;
};

// Workgroup -> C tile. Workgroups are dealt to the 8 XCDs round-robin; this
// gives each XCD a contiguous run of tile ids, and runs of GM_GROUP tile rows
// sweep the tile columns together, so an XCD's L2 sees the same B columns
// and A rows reused.
VH_DEV void gm_tile_of(int bid, int nblk, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int per = nblk / 8, rem = nblk % 8;
  const int x = bid % 8, local = bid / 8;
  const int t = x * per + (x < rem ? x : rem) + local;
  const int span = GM_GROUP * tiles_n;
  const int first = (t / span) * GM_GROUP;
  const int gsize = tiles_m - first < GM_GROUP ? tiles_m - first : GM_GROUP;
  const int in = t % span;
  tm = first + in % gsize;
  tn = in / gsize;
}

// The launch's causal mode: a.causal, unless a device flag says the product is dense.
VH_DEV int gm_causal(const GemmArgs& a) { return (a.causal_flag && *a.causal_flag == 0) ? 0 : a.causal; }
// The addend: under a device flag that says causal, E is the attention's mask,
// whose allowed entries are +-0 and whose masked ones the causal form skips, so
// it is not added (as a caller passing causal = 1 drops it).
VH_DEV const float* gm_addend(const GemmArgs& a) {
  return (a.causal_flag && *a.causal_flag != 0) ? nullptr : a.E;
}

// The epilogue of one output element from its product sum v: the raw partial
// under split-K (raw), else alpha v (+ E[m, n]) (+ old = out[m, n]).
VH_DEV float gm_finish(const GemmArgs& a, const float* E, bool raw, float v, int64_t m, int64_t n, float old) {
  if (raw) return v;
  v = v * a.alpha;
  if (E) v = v + E[m * a.sem + n * a.sen];
  if (a.accumulate) v = old + v;
  return v;
}

// A wave's MT x NTW matrix-core tiles of the T-row tile at (m0, n0) straight from
// its accumulators: register r of a 32 x 32 tile holds row 8*(r/4) + 4*h + r%4,
// column li; elements outside M x N are dropped. NT: streaming (nontemporal)
// stores, which do not allocate the written lines in L2.
template <int MT, int NTW, bool NT = false>
VH_DEV void gm_store_direct(const GemmArgs& a, const vh_f32x16 (&acc)[MT][NTW], float* out, int64_t ldo,
                            const float* E, bool raw, int64_t m0, int64_t n0, int T, int wm, int wn, int li, int h) {
  if (m0 + T <= a.M && n0 + NTW * 64 <= a.N && (raw || !a.accumulate) && (raw || !E || a.sem == 0)) {
    // A whole tile that reads nothing back but a bias row: the stores go out back
    // to back (a conditional load of C among them makes each wait for all earlier
    // stores, as the memory counter covers both).
    const float alpha = raw ? 1.0f : a.alpha;
    const bool bias = !raw && E;
    float* base = out + (m0 + wm * (MT * 32) + 4 * h) * ldo + n0 + wn * (NTW * 32) + li;
    float eb[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) eb[nt] = bias ? E[(n0 + wn * (NTW * 32) + nt * 32 + li) * a.sen] : 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float* cp = base + (mt * 32 + 8 * (r >> 2) + (r & 3)) * ldo + nt * 32;
          float v = raw ? acc[mt][nt][r] : acc[mt][nt][r] * alpha;
          if (bias) v = v + eb[nt];
          if constexpr (NT)
            __builtin_nontemporal_store(v, cp);
          else
            *cp = v;
        }
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      const int64_t n = n0 + wn * (NTW * 32) + nt * 32 + li;
      // (the old C of a whole column goes out before its stores, see above)
      float old[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm * (MT * 32) + mt * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        old[r] = a.accumulate && !raw && m < a.M && n < a.N ? out[m * ldo + n] : 0.0f;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm * (MT * 32) + mt * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (m < a.M && n < a.N) {
          float* cp = out + m * ldo + n;
          const float v = gm_finish(a, E, raw, acc[mt][nt][r], m, n, old[r]);
          if constexpr (NT)
            __builtin_nontemporal_store(v, cp);
          else
            *cp = v;
        }
      }
    }
  }
}

// Buffer resource of `bytes` bytes from `org`, clamped to [0, 2^32 - 1], and a
// 128-bit load through it (4-byte alignment is enough; each dword past the end
// reads 0 on its own).
VH_DEV __amdgpu_buffer_rsrc_t gm_rsrc(const float* org, int64_t bytes) {
  uint32_t hi = (uint32_t)((uint64_t)bytes >> 32), lo = (uint32_t)bytes;
  asm("" : "+s"(hi), "+s"(lo));  // keeps the compiler from joining the halves into a vector compare
  const uint32_t nrec = (int32_t)hi < 0 ? 0u : (hi != 0 ? 0xFFFFFFFFu : lo);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(org), (short)0, (int)nrec, 0x00020000);
}
VH_DEV vh_f4 gm_bload(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(vh_f4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// The tiled product on the bf16 instruction (split3.h): a 256-thread workgroup
// computes a T x T tile of C (T = 128 or 64), its four waves T/2 x T/2 quadrants as
// NW x NW matrix-core tiles of 32 x 32. K advances in tiles of 32: each thread
// brings T/64 pieces of eight consecutive k of a row of each operand (gt_load),
// splits them and writes the parts' 16-byte fragments to LDS, laid out [part][k
// eighth][row]. A k tile's products are summed on their own (tt, 12 roundings of
// the small sum) and then added to acc in f32, so an element sees one rounding
// per 32 k at its own size: measured at K = 768, 1.3e-7 of the result against 5.0e-7
// on the f32 instruction.
//
// T = 64 runs two LDS stages, one barrier per k tile, and loads two k tiles ahead:
// for products whose few tiles leave the chip's latency exposed. T = 128 runs one
// stage (50 KB, so that two workgroups share a CU and cover each other's barriers
// and loads) and loads one k tile ahead.
//
// BUF operands come through buffer loads, whose bounds make rows past the
// operand's last element read 0 and which need only 4-byte alignment; the others
// (leading dimensions whose tile reads pass 2^32 bytes) element by element.
template <bool A_KC, bool A_BUF, bool B_KC, bool B_BUF, int T>
struct GemmTile {
  static constexpr int HS = T * 4 + 16, OP = 12 * HS;  // dwords per k eighth (64 bytes of padding), per operand
  static constexpr int D = T == 64 ? 2 : 1;            // LDS stages
  using Lds = uint32_t[D][2][OP];
  // The staging registers (a k tile of each operand), and where a tile's first k tile is.
  struct Regs {
    vh_f4 a[D][T / 64][2], b[D][T / 64][2];
  };
  struct Origin {
    const float *A, *B;
    int64_t m0, n0;
  };
  // C tile (tm, tn) of batch `bat`, or its raw partial over K range `kr` of a.ksplit.
  // STREAM (T = 128, no split): R holds the tile's first k tile already, and the last k
  // step loads the one at `next` (null: none) into it; streaming stores.
  template <bool STREAM = false>
  static VH_DEV void run(const GemmArgs& a, Lds& L, int tm, int tn, int64_t bat, int kr, int causal, Regs& R,
                         const Origin* next = nullptr);
  static VH_DEV Origin origin(const GemmArgs& a, int tm, int tn, int64_t bat) {
    const int64_t b1 = bat / a.nb2, b2 = bat % a.nb2;
    return Origin{a.A + b1 * a.sa1 + b2 * a.sa2, a.B + b1 * a.sb1 + b2 * a.sb2, (int64_t)tm * T, (int64_t)tn * T};
  }
  static VH_DEV int k8_of(bool kc, int u) { return kc ? threadIdx.x & 3 : ((threadIdx.x >> 6) + 4 * u) & 3; }
  // The pieces of the k tile at k0 of rows r0 .. (R of them, K long) into v.
  template <bool KC, bool BUF>
  static VH_DEV void load(const float* X, int64_t ld, int64_t r0, int64_t R, int64_t k0, int64_t K,
                          vh_f4 (&v)[T / 64][2]);
  static VH_DEV void load_tile(const GemmArgs& a, const Origin& o, int64_t k0, Regs& R, int set) {
    load<A_KC, A_BUF>(o.A, a.lda, o.m0, a.M, k0, a.K, R.a[set]);
    load<B_KC, B_BUF>(o.B, a.ldb, o.n0, a.N, k0, a.K, R.b[set]);
  }
};

template <bool A_KC, bool A_BUF, bool B_KC, bool B_BUF, int T>
VH_DEV void gemm_tile_impl(const GemmArgs& a) {
  using Tile = GemmTile<A_KC, A_BUF, B_KC, B_BUF, T>;
  __shared__ __attribute__((aligned(1024))) typename Tile::Lds L;
  int tm, tn;
  int64_t bat = blockIdx.y;  // batch index (both batch dims), or the K range
  const int causal = gm_causal(a);
  if (causal >= 2 && a.ksplit <= 1) {
    // The k range grows with the tile row (k <= m) or shrinks (k >= m): deal
    // the workgroups longest first across all batches, so the last ones to
    // start are short (the launch order is x fastest, then y).
    const int64_t lin = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int64_t rank = lin / gridDim.y;
    bat = lin % gridDim.y;
    const int row = (int)(rank / a.tiles_n);
    tm = causal == 2 ? a.tiles_m - 1 - row : row;
    tn = (int)(rank % a.tiles_n);
  } else {
    gm_tile_of(blockIdx.x, gridDim.x, a.tiles_m, a.tiles_n, tm, tn);
  }
  typename Tile::Regs R;
  Tile::run(a, L, tm, tn, bat, (int)blockIdx.y, causal, R);
}

// The persistent form for dense products: the grid is at most the chip's
// resident workgroups, each walking the (tile, K range) pairs of all batches.
template <bool A_KC, bool B_KC, int T>
VH_DEV void gemm_tile_walk(const GemmArgs& a) {
  using Tile = GemmTile<A_KC, true, B_KC, true, T>;
  __shared__ __attribute__((aligned(1024))) typename Tile::Lds L;
  const int tiles = a.tiles_m * a.tiles_n;
  const int64_t items = (int64_t)tiles * (a.ksplit > 1 ? a.ksplit : a.nbat);
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    int tm, tn;
    gm_tile_of((int)(it % tiles), tiles, a.tiles_m, a.tiles_n, tm, tn);
    typename Tile::Regs R;
    Tile::run(a, L, tm, tn, it / tiles, (int)(it / tiles), 0, R);
    __syncthreads();  // the next item stages into the LDS this one read
  }
}

template <bool A_KC, bool A_BUF, bool B_KC, bool B_BUF, int T>
template <bool KC, bool BUF>
VH_DEV void GemmTile<A_KC, A_BUF, B_KC, B_BUF, T>::load(const float* X, int64_t ld, int64_t r0, int64_t R, int64_t k0,
                                                        int64_t K, vh_f4 (&v)[T / 64][2]) {
  const uint32_t tid = threadIdx.x, w = tid >> 6, q4 = (tid & 63) >> 4, c4 = tid & 15;
  if constexpr (BUF) {
    const auto r = gm_rsrc(X + (KC ? r0 * ld + k0 : k0 * ld + r0),
                           (KC ? (R - 1 - r0) * ld + K - k0 : (K - 1 - k0) * ld + R - r0) * 4);
    const uint32_t ld4 = (uint32_t)ld * 4u;
#pragma unroll
    for (int u = 0; u < T / 64; ++u) {
      const uint32_t o = KC ? ((tid >> 2) + 64u * u) * ld4 + k8_of(true, u) * 32u
                            : (8u * k8_of(false, u) + 2u * q4) * ld4 + (((w + 4u * u) >> 2) * 64u + 4u * c4) * 4u;
      v[u][0] = gm_bload(r, o);
      v[u][1] = gm_bload(r, o + (KC ? 16u : ld4));
    }
  } else {
#pragma unroll
    for (int u = 0; u < T / 64; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int64_t r = r0 + (KC ? (tid >> 2) + 64 * u : ((w + 4 * u) >> 2) * 64 + 4 * c4 + (e & 3));
        const int64_t k = k0 + 8 * k8_of(KC, u) + (KC ? e : 2 * q4 + (e >> 2));
        v[u][e >> 2][e & 3] = r < R && k < K ? X[KC ? r * ld + k : k * ld + r] : 0.0f;
      }
  }
}

template <bool A_KC, bool A_BUF, bool B_KC, bool B_BUF, int T>
template <bool STREAM>
VH_DEV void GemmTile<A_KC, A_BUF, B_KC, B_BUF, T>::run(const GemmArgs& a, Lds& L, int tm, int tn, int64_t bat, int kr,
                                                       int causal, Regs& R, const Origin* next) {
  static_assert((T == 128 || T == 64) && !(STREAM && T == 64), "tile");
  constexpr int NW = T / 64, U = T / 64;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1, li = lane & 31, h = lane >> 5, q4 = lane >> 4, c4 = lane & 15;
  const int64_t m0 = (int64_t)tm * T, n0 = (int64_t)tn * T;
  if (causal == 1 && n0 > m0 + T - 1) return;  // the whole tile is masked

  const bool split = a.ksplit > 1;
  const int64_t b1 = split ? 0 : bat / a.nb2, b2 = split ? 0 : bat % a.nb2;
  const float* A = a.A + b1 * a.sa1 + b2 * a.sa2;
  const float* B = a.B + b1 * a.sb1 + b2 * a.sb2;
  float* C = a.C + b1 * a.sc1 + b2 * a.sc2;

  int64_t kb = 0, ke = a.K;
  if (causal == 2) ke = m0 + T < a.K ? m0 + T : a.K;
  if (causal == 3) kb = (m0 / GM_TK) * GM_TK;
  if (split) {
    kb = (int64_t)kr * a.kchunk;
    ke = kb + a.kchunk < a.K ? kb + a.kchunk : a.K;
  }
  // K <= 8 runs on the f32 instruction (below): a single product there is correctly
  // rounded, the split's is up to 0.94 ulp off (1.9 u, measured over 65536), which
  // more products' own roundings cover.
  const bool tiny = a.K <= 8;
  const int steps = ke > kb && !tiny ? (int)((ke - kb + GM_TK - 1) / GM_TK) : 0;

  // Piece u of a thread: row and k eighth, and its dword in an LDS part. k-contiguous:
  // four threads cover a row's 128 bytes. Row-contiguous: wave w takes 64-row
  // block (w + 4 u) / 4 and k eighth (w + 4 u) % 4; lane 16 q + c loads rows 4 c .. 4 c + 3
  // at k = 2 q and 2 q + 1, and a transpose across the lanes' q leaves it all eight k of
  // row 4 c + q (at LDS piece 16 q + (c + 4 q) % 16 of the block, which the writes and
  // the fragment reads of 16 lanes both meet without bank conflicts).
  auto lds_of = [&](bool kc, int u) {
    const int piece = kc ? (tid >> 2) + 64 * u : ((w + 4 * u) >> 2) * 64 + 16 * q4 + ((c4 + 4 * q4) & 15);
    return k8_of(kc, u) * HS + 4 * piece;
  };
  const GmFlag<A_KC> akc{};
  const GmFlag<B_KC> bkc{};
  // Factors of the pieces: S3_SCALE, negative in every other group of 32 rows of A and
  // columns of B, and in every other k tile of A: the matrix core's sums drift
  // towards minus infinity by what they round off (gemm_split.h), which then cancels
  // along K and over rows and columns.
  const float fsa = (A_KC ? tid >> 7 : c4 >> 3) & 1 ? -S3_SCALE : S3_SCALE;
  const float fsb = (B_KC ? tid >> 7 : c4 >> 3) & 1 ? -S3_SCALE : S3_SCALE;
  auto k_sign = [](int64_t k0) { return k0 & GM_TK ? -1.0f : 1.0f; };
  // Splits the staged pieces into LDS; k past K (what the loads returned there is
  // another row's) as zeros, in both operands.
  auto stage = [&](auto kcv, const vh_f4 (&v)[U][2], uint32_t* S, int64_t k0, float f) {
    constexpr bool KC = decltype(kcv)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float x[8];
      if constexpr (KC) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = v[u][e >> 2][e & 3];
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const vh_u4 t4 = __builtin_bit_cast(vh_u4, v[u][e]);
          uint32_t t[4] = {t4[0], t4[1], t4[2], t4[3]};
          s3_transpose4(t);
#pragma unroll
          for (int j = 0; j < 4; ++j) x[2 * j + e] = __builtin_bit_cast(float, t[j]);
        }
      }
      if (k0 + GM_TK > a.K) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = k0 + 8 * k8_of(KC, u) + e < a.K ? x[e] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= f;
      vh_u4 p[3];
      s3_split8(x, p);
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<vh_u4*>(S + t * 4 * HS + lds_of(KC, u)) = p[t];
    }
  };
  auto lds_barrier = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  vh_f32x16 acc[NW][NW], tt[NW][NW];
#pragma unroll
  for (int i = 0; i < NW; ++i)
#pragma unroll
    for (int j = 0; j < NW; ++j) acc[i][j] = vh_f32x16{};
  // Row 32 g + li of an operand's tile: its LDS piece.
  const int lt = 16 * (li & 3) + (((li >> 2) + 4 * (li & 3)) & 15);
  auto piece = [&](bool kc, int g) { return kc ? 32 * g + li : 64 * (g >> 1) + (g & 1 ? lt ^ 8 : lt); };
  vh_u4 fa[2][NW][3], fb[2][NW][3];
  auto frags = [&](const uint32_t* SA, const uint32_t* SB, int kk) {
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const int o = (4 * t + 2 * kk + h) * HS;
        fa[kk][i][t] = *reinterpret_cast<const vh_u4*>(SA + o + 4 * piece(A_KC, wm * NW + i));
        fb[kk][i][t] = *reinterpret_cast<const vh_u4*>(SB + o + 4 * piece(B_KC, wn * NW + i));
      }
  };
  auto products = [&](int kk) {
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < NW; ++j)
          tt[i][j] = s3_mfma(fa[kk][i][S3_PA(t)], fb[kk][j][S3_PB(t)], kk || t ? tt[i][j] : vh_f32x16{});
  };
  auto add = [&](float sg) {
    if (((wm + wn) * NW) & 1) sg = -sg;
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int j = 0; j < NW; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(tt[i][j][r], (i ^ j) & 1 ? -sg : sg, acc[i][j][r]);
  };
  const Origin og{A, B, m0, n0};
  // Loads past the last k tile fetch it again (every load stays in the range).
  auto k_at = [&](int st) { return kb + (int64_t)(st < steps ? st : steps - 1) * GM_TK; };
  if (steps > 0) {
    if constexpr (D == 2) {
      // Two stages: k tile st is multiplied from one while st + 1 is split into the
      // other (free since the barrier: its readers have passed it), its registers
      // then reloaded with st + 3.
      load_tile(a, og, k_at(0), R, 0);
      load_tile(a, og, k_at(1), R, 1);
      stage(akc, R.a[0], L[0][0], k_at(0), fsa * k_sign(kb));
      stage(bkc, R.b[0], L[0][1], k_at(0), fsb);
      load_tile(a, og, k_at(2), R, 0);
      for (int st = 0; st < steps; st += 2) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          if (st + d < steps) {
            lds_barrier();
            frags(L[d][0], L[d][1], 0);
            frags(L[d][0], L[d][1], 1);
            products(0);
            stage(akc, R.a[d ^ 1], L[d ^ 1][0], k_at(st + d + 1), fsa * k_sign(k_at(st + d + 1)));
            products(1);
            stage(bkc, R.b[d ^ 1], L[d ^ 1][1], k_at(st + d + 1), fsb);
            load_tile(a, og, k_at(st + d + 3), R, d ^ 1);
            add(k_sign(k_at(st + d)));
          }
        }
      }
    } else {
      if constexpr (!STREAM) load_tile(a, og, k_at(0), R, 0);
      for (int st = 0; st < steps; ++st) {
        stage(akc, R.a[0], L[0][0], k_at(st), fsa * k_sign(k_at(st)));
        stage(bkc, R.b[0], L[0][1], k_at(st), fsb);
        if (STREAM && next && st + 1 == steps)
          load_tile(a, *next, 0, R, 0);
        else
          load_tile(a, og, k_at(st + 1), R, 0);
        lds_barrier();
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          frags(L[0][0], L[0][1], kk);
          products(kk);
        }
        add(k_sign(k_at(st)));
        lds_barrier();
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NW; ++i)
#pragma unroll
    for (int j = 0; j < NW; ++j) acc[i][j] *= S3_UNSCALE;
  // On the f32 instruction, straight from memory: all of a tiny product, or, a 32 x 32 tile
  // at a time, the infinities and NaN of another (see split3.h). Rows past M (columns
  // past N) and k past the range read as zero.
  auto a_at = [&](int64_t m, int64_t k) { return m < a.M && k < ke ? A[A_KC ? m * a.lda + k : k * a.lda + m] : 0.0f; };
  auto b_at = [&](int64_t n, int64_t k) { return n < a.N && k < ke ? B[B_KC ? n * a.ldb + k : k * a.ldb + n] : 0.0f; };
  if (tiny) {
#pragma nounroll
    for (int64_t k = kb; k < ke; k += 2) {
      float x[NW], y[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        x[i] = a_at(m0 + wm * (T / 2) + 32 * i + li, k + h);
        y[i] = b_at(n0 + wn * (T / 2) + 32 * i + li, k + h);
      }
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < NW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], y[j], acc[i][j], 0, 0, 0);
    }
  } else if (s3_nonfinite(acc)) {
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const int64_t mt = m0 + wm * (T / 2) + 32 * i, n = n0 + wn * (T / 2) + 32 * j + li;
        const uint32_t bad = s3_nonfinite_regs(acc[i][j], a.M - mt - 4 * h, a.N - n);
        if (__builtin_amdgcn_ballot_w64(bad != 0) == 0) continue;
        vh_f32x16 t{};
#pragma nounroll
        for (int64_t k = kb; k < ke; k += 2)
          t = __builtin_amdgcn_mfma_f32_32x32x2f32(a_at(mt + li, k + h), b_at(n, k + h), t, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = bad >> r & 1 ? t[r] : acc[i][j][r];
      }
  }

  float* out = split ? a.ws + (int64_t)kr * a.M * a.N : C;
  const float* E0 = gm_addend(a);
  const float* E = !split && E0 ? E0 + b1 * a.se1 + b2 * a.se2 : nullptr;
  gm_store_direct<NW, NW, STREAM>(a, acc, out, split ? a.N : a.ldc, E, split, m0, n0, T, wm, wn, li, h);
}

// Persistent form for batched products with a short k range (attention's
// scores q k^T and dP = dO v^T: K = Dk = 64, 2 k tiles per C tile). Launched
// as one workgroup per resident slot (a multiple of 8), each walks a list of
// 128 x 128 C tiles as one continuous k loop: the last k step of a tile loads the
// first k tile of the next one, so its global loads are in flight under the
// current tile's products and epilogue instead of exposed at the start of a
// short-lived workgroup. Work items are the live tiles of every batch, batch
// major (causal 1: the tiles with tn <= tm, which with tiles_n >= tiles_m are
// T (T + 1) / 2 for T = tiles_m); XCD x (= workgroup id % 8, the hardware's
// round-robin) takes the x-th contiguous eighth of the items, so one XCD works
// on one or two batches at a time and its L2 holds their operands. No split,
// causal 0 or 1 only (the host guarantees both).
//
// 192 x [1024, 64] x [64, 1024], causal (453 MB of live tiles): 172 us on the f32
// instruction (92 us of it matrix work at that instruction's peak), 150 on the
// three-part split, 3.0 TB/s written. The instruction's rate no longer bounds it:
// the splits, LDS traffic and stores of each 64-deep tile do, two workgroups per
// CU (registers) covering each other's.
template <bool A_KC, bool B_KC>
VH_DEV void gemm_tile_stream(const GemmArgs& a) {
  using Tile = GemmTile<A_KC, true, B_KC, true, 128>;
  __shared__ __attribute__((aligned(1024))) typename Tile::Lds L;
  const int causal = gm_causal(a);
  const int64_t live = causal == 1 ? (int64_t)a.tiles_m * (a.tiles_m + 1) / 2 : (int64_t)a.tiles_m * a.tiles_n;
  const int64_t total = live * a.nbat;
  const int nloc = (int)(gridDim.x / 8), x = (int)(blockIdx.x % 8);
  const int64_t per = (total + 7) / 8;
  const int64_t end = (x + 1) * per < total ? (x + 1) * per : total;
  int64_t item = x * per + (int64_t)(blockIdx.x / 8);
  if (item >= end) return;

  auto decode = [&](int64_t it, int& tm, int& tn, int64_t& bat) {
    bat = it / live;
    const int64_t u = it % live;
    if (causal == 1) {  // u = tm (tm + 1) / 2 + tn, tn <= tm
      int64_t t = (int64_t)((sqrtf(8.0f * (float)u + 1.0f) - 1.0f) * 0.5f);
      while (t * (t + 1) / 2 > u) --t;
      while ((t + 1) * (t + 2) / 2 <= u) ++t;
      tm = (int)t;
      tn = (int)(u - t * (t + 1) / 2);
    } else {
      tm = (int)(u / a.tiles_n);
      tn = (int)(u % a.tiles_n);
    }
  };
  int tm, tn;
  int64_t bat;
  decode(item, tm, tn, bat);
  typename Tile::Regs R;
  Tile::load_tile(a, Tile::origin(a, tm, tn, bat), 0, R, 0);
  for (;;) {
    const int64_t nit = item + nloc;
    const bool more = nit < end;
    int tm2 = tm, tn2 = tn;
    int64_t bat2 = bat;
    if (more) decode(nit, tm2, tn2, bat2);
    const typename Tile::Origin next = Tile::origin(a, tm2, tn2, bat2);
    Tile::template run<true>(a, L, tm, tn, bat, 0, causal, R, &next);
    if (!more) break;
    item = nit;
    tm = tm2;
    tn = tn2;
    bat = bat2;
  }
}

// C[m, n] = epilogue(sum over y of ws[y][m][n], y ascending): the split-K
// partials in a fixed order, so the result does not depend on timing.
VH_DEV void gemm_reduce_impl(const GemmReduceArgs& a) {
  const int64_t total = a.M * a.N;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    const int64_t m = i / a.N, n = i % a.N;
    float s = a.ws[i];
    for (int y = 1; y < a.ksplit; ++y) s += a.ws[(int64_t)y * total + i];
    float v = s * a.alpha;
    if (a.E) v = v + a.E[m * a.sem + n * a.sen];
    float* cp = a.C + m * a.ldc + n;
    if (a.accumulate) v = *cp + v;
    *cp = v;
  }
}
