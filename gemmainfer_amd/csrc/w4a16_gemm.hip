// W4A16 linear for more than 16 token rows on gfx950: C[M, N] = A[M, K] @
// dequant(B), the projections of a prompt (and of batches past the decode
// kernels' 16 rows), for bf16 and fp16 activations.
//
// Reference behaviour restated (paths relative to the GemmaInfer repo):
//   csrc/marlin.cu:207-260, :764-842 (M > 8: one row per block row there, the
//   weights re-read for every row), csrc/pybind.cpp:46-85 (semantics),
//   gemmainfer/kernels/activations.py:21-34 (gated MLP).
//
// Two launches:
//   order  the token rows into operand fragments: the 64 x 16 bytes one wave
//          loads as the A operand of one 16-row x 32-k matrix-core product,
//          1 KB in a row, k order of the unpacked words; and, for bf16, -24
//          times the sum of each row over each unit of k (the offset of the
//          16 + q operands).  One pass over A, so that the products' kernel
//          stages A without touching it.
//   gemm   64 rows x 256 columns per workgroup (see below)
//
// Rows past M and k past K are zero fragments: the products need no bounds.
// Calls whose grid of such tiles would not fill the chip run a kernel of
// smaller tiles and a K split instead, in one launch (64 x 2816 x 4096: 14.2
// us, bf16, kernel trace).

#include "../../include/gemmainfer_amd.h"
#include "gi_common.h"
#include "gi_internal.h"
#include "moe_shared.h"

namespace gi {

namespace {

using moe::f32x4_t;
constexpr int kGmThreads = 256;
constexpr int kGmRows = 64;      // token rows per workgroup
constexpr int kGmCols = 256;     // columns per workgroup (64 per wave)
constexpr int kGmRT = kGmRows / 16;
constexpr int kGmChunk = 4;      // k blocks (of 32) staged per barrier

struct GmArgs {
  const uint4* xf;      // [row tiles][KBp][64] operand fragments
  const float* off;     // [row blocks][units][64 rows]: -24 * sum of the row over the unit (bf16)
  int M, K, KBp;        // KBp: k blocks padded to whole chunks
  int gs, rb, total;    // rb row blocks; total workgroups
  int c8;               // every C is 8-byte aligned (a view may start at any element)
  float cap;
  GemmSeg seg[kMaxGemmSegs];
};

struct GmOrderArgs {
  const uint16_t* A;
  uint4* xf;
  float* off;
  int M, K, KBp, units;
};

// One wave per (16-row tile, unit of KPG k blocks).
template <int KPG, bool F16>
__global__ __launch_bounds__(256) void gemm_order_kernel(GmOrderArgs a) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int lq = lane >> 4, lr = lane & 15;
  const int u = blockIdx.x * 4 + wave, rt = blockIdx.y;
  if (u >= a.units) return;
  const int row = 16 * rt + lr;
  const bool row_ok = row < a.M;
  const uint16_t* src = a.A + (size_t)(row_ok ? row : 0) * a.K;
  uint4 d[KPG];
#pragma unroll
  for (int s = 0; s < KPG; ++s) {
    const int k = 32 * (u * KPG + s) + 8 * lq;
    const bool ok = row_ok && k < a.K;
    d[s] = *(const uint4*)(src + (ok ? k : 0));
    if (!ok) d[s] = make_uint4(0u, 0u, 0u, 0u);
  }
  float b = 0.f;
#pragma unroll
  for (int s = 0; s < KPG; ++s) {
    a.xf[((size_t)rt * a.KBp + u * KPG + s) * kWave + lane] = moe::mfma_k_order(d[s]);
    if constexpr (!F16) b += q4_bias(d[s]);
  }
  if constexpr (!F16) {
    b += __shfl_xor(b, 16, kWave);
    b += __shfl_xor(b, 32, kWave);
    if (lane < 16) a.off[((size_t)(rt / kGmRT) * a.units + u) * kGmRows + row % kGmRows] = b;
  }
}

// Four 16-bit results in a row (N is a multiple of 4).
__device__ __forceinline__ void gm_store4(uint16_t* c, uint2 v, int c8) {
  if (c8) {
    *(uint2*)c = v;
  } else {
    c[0] = (uint16_t)v.x;
    c[1] = (uint16_t)(v.x >> 16);
    c[2] = (uint16_t)v.y;
    c[3] = (uint16_t)(v.y >> 16);
  }
}

// The products.  A workgroup of 4 waves owns 64 rows x 256 columns over all of
// K; wave w 64 of the columns: lane (lq, lr) loads the 16 bytes of columns
// 4lr..4lr+3 at packed row 4kb + lq, i.e. the B operands of four 16-column
// products, so each word is loaded and unpacked by one wave and serves 64
// rows.  The A fragments of a chunk (4 k blocks, 16 KB) are staged in LDS,
// two chunk buffers, one barrier per chunk; words, scales and fragments are
// loaded one chunk ahead.
//
// What bounds it: instruction issue.  A row tile's stage (64 k) is 8 products
// of 16 cycles each and, beside them, 16 scaled sums and 16 operations of the
// next unit's unpack, 4 cycles each; at 2048 rows, K 2816, N 8192 (118 us in a
// kernel trace, 799 TFLOP/s, and 8 us for the order launch) the matrix cores
// are busy 38% of the time and the VALU issues 56% of it.  So everything
// is laid out for fewer and overlapped VALU operations: the offset enters as
// the products' starting value (no product and no add of its own), a stage's
// sums are taken under the next stage's products, the unpack is spread over
// the stages, and the order of each stage is pinned (left to itself the
// compiler loads a fragment and waits for it, stage by stage, and drains every
// load at the loop's head: 2048 x 2816 x 8192 169.7 -> 109.4 us, the fastest
// whole calls of one box; 64 x 2816 x 4096, which now takes the small kernel,
// 59.7 -> 32.4 us).
template <int KPG, bool F16, bool GATED>
__global__ __launch_bounds__(kGmThreads, 2) void gemm_kernel(GmArgs a) {
  constexpr int kUnits = kGmChunk / KPG;   // units per chunk
  constexpr int kStages = kUnits * kGmRT;  // (unit, row tile) pairs per chunk
  constexpr int kWords = 4 * KPG;          // words per unit and lane
  __shared__ uint4 xs[2][kGmRT][kGmChunk][kWave];
  __shared__ float os[2][kGmThreads / kWave][kGmRows];  // [buffer][unit of the chunk]
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, lr = lane & 15;
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles
  // (row blocks fastest), so the words of a column tile and the fragments
  // meet in one L2
  const int xcd = blockIdx.x & 7, base = a.total >> 3, rem = a.total & 7;
  const int t = xcd * base + min(xcd, rem) + (int)(blockIdx.x >> 3);
  int ct = t / a.rb;
  const int rb = t - ct * a.rb;
  GemmSeg sg = a.seg[0];
  if constexpr (GATED) {
    if (wave >= 2) sg = a.seg[1];
  } else {
#pragma unroll
    for (int i = 1; i < kMaxGemmSegs; ++i)
      if (ct >= a.seg[i].tile0) sg = a.seg[i];
    ct -= sg.tile0;
  }
  const int col = (GATED ? ct * (kGmCols / 2) + (wave & 1) * 64 : ct * kGmCols + wave * 64) + 4 * lr;
  // columns past N read the last four (their results are not stored)
  const int colr = min(col, sg.N - 4);
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(sg.B, (uint32_t)((size_t)(a.K >> 3) * sg.N * 4));
  const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(sg.S, (uint32_t)((size_t)sg.G * sg.N * 2));
  // k past the last scale group (the longer table's of GATED) is dropped: the
  // fragments and offsets end there and read zeros beyond, since a zero scale
  // alone would make NaN of an infinity or NaN in a dropped column
  const int units = a.KBp / KPG, upg = a.gs / (32 * KPG);  // units of k; units per scale group
  const int live = min(units, (GATED ? max(a.seg[0].G, a.seg[1].G) : sg.G) * upg);
  const __amdgpu_buffer_rsrc_t rx =
      buffer_rsrc(a.xf + (size_t)(rb * kGmRT + wave) * a.KBp * kWave, (uint32_t)(live * KPG) * kWave * 16u);
  const __amdgpu_buffer_rsrc_t ro =
      buffer_rsrc(a.off + (size_t)rb * units * kGmRows, F16 ? 0u : (uint32_t)(live * kGmRows) * 4u);
  const uint32_t wstep = (uint32_t)sg.N * 16u;
  const uint32_t wbase = ((uint32_t)lq * (uint32_t)sg.N + (uint32_t)colr) * 4u;
  auto wload = [&](int kb) {
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rw, wbase + (uint32_t)kb * wstep, 0, 0);
    return make_uint4(v.x, v.y, v.z, v.w);
  };
  const uint32_t sbase = (uint32_t)colr * 2u, sstep = (uint32_t)sg.N * 2u;
  auto sload = [&](int u) {
    // groups past the scales tensor read zeros
    const int g = u / upg;
    const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rs, g < sg.G ? sbase + (uint32_t)g * sstep : 0xFFFFFFF0u, 0, 0);
    return make_uint2(v.x, v.y);
  };

  const uint32_t mq = moe::q4_magic_t<F16>();
  const f32x4_t zf = {0.f, 0.f, 0.f, 0.f};
  f32x4_t y[kGmRT][4];
#pragma unroll
  for (int rt = 0; rt < kGmRT; ++rt)
#pragma unroll
    for (int q = 0; q < 4; ++q) y[rt][q] = zf;

  const int nch = a.KBp / kGmChunk;
  // the next chunk's fragments of row tile `wave` and its offsets (past the
  // last chunk: zeros, no memory access)
  u32x4_t ar[kGmChunk];
  uint32_t orr;
  auto aload = [&](int c) {
#pragma unroll
    for (int j = 0; j < kGmChunk; ++j)
      ar[j] = __builtin_amdgcn_raw_buffer_load_b128(rx, (uint32_t)((c * kGmChunk + j) * kWave + lane) * 16u, 0, 0);
    if constexpr (!F16)
      orr = __builtin_amdgcn_raw_buffer_load_b32(ro, (uint32_t)((c * kUnits + wave) * kGmRows + lane) * 4u, 0, 0);
  };
  auto astore = [&](int b) {
#pragma unroll
    for (int j = 0; j < kGmChunk; ++j) *(u32x4_t*)&xs[b][wave][j][lane] = ar[j];
    if constexpr (!F16) os[b][wave][lane] = __uint_as_float(orr);
  };
  uint4 wr[kGmChunk];      // words of the chunk being multiplied, then of the next
  uint2 sr[kUnits];        // scales likewise
  uint32_t B[2][kWords][4];  // unpacked operands: this unit's and the next's
  f32x4_t D[2][4];         // a stage's products, and the previous stage's
  float sc[2][4];
  auto unpack = [&](int p, int i, uint32_t w) {
    const uint4 o = moe::q4_operand_t<F16>(w, mq);
    B[p][i][0] = o.x;
    B[p][i][1] = o.y;
    B[p][i][2] = o.z;
    B[p][i][3] = o.w;
  };
  auto word = [&](int j, int q) { return q == 0 ? wr[j].x : q == 1 ? wr[j].y : q == 2 ? wr[j].z : wr[j].w; };
  auto scales = [&](int p, uint2 v) {
    sc[p][0] = moe::sc_lo<F16>(v.x);
    sc[p][1] = moe::sc_hi<F16>(v.x);
    sc[p][2] = moe::sc_lo<F16>(v.y);
    sc[p][3] = moe::sc_hi<F16>(v.y);
    // taken out of the loaded words here, so that those can be loaded again
    // (left to itself the compiler unpacks at the use and copies the words)
#pragma unroll
    for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(sc[p][q]));
  };
  aload(0);
#pragma unroll
  for (int j = 0; j < kGmChunk; ++j) wr[j] = wload(j);
#pragma unroll
  for (int u = 0; u < kUnits; ++u) sr[u] = sload(u);
  astore(0);
  aload(1);
#pragma unroll
  for (int i = 0; i < kWords; ++i) unpack(0, i, word(i / 4, i % 4));
#pragma unroll
  for (int j = 0; j < KPG; ++j) wr[j] = wload(kGmChunk + j);
  scales(0, sr[0]);
  sr[0] = sload(kUnits);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    D[1][q] = zf;
    sc[1][q] = 0.f;
  }
#pragma unroll 1
  for (int c = 0; c < nch; ++c) {
    lds_barrier();  // chunk c is staged; every reader of chunk c - 1 is done
    const int b = c & 1;
    uint4 A[2][KPG];
    f32x4_t O[2];
    auto frag = [&](int st, int p) {
      const int u = st / kGmRT, rt = st % kGmRT;
#pragma unroll
      for (int s = 0; s < KPG; ++s) A[p][s] = xs[b][rt][u * KPG + s][lane];
      O[p] = zf;
      if constexpr (!F16) O[p] = *(const f32x4_t*)&os[b][u][16 * rt + 4 * lq];
    };
    frag(0, 0);
    astore((c + 1) & 1);
    aload(c + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < kStages; ++st) {
      const int u = st / kGmRT, rt = st % kGmRT, p = st & 1, up = u & 1;
      if (st + 1 < kStages) frag(st + 1, p ^ 1);
      // this stage's products
#pragma unroll
      for (int s = 0; s < KPG; ++s)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t* o = B[up][4 * s + q];
          D[p][q] = moe::mfma_act<F16>(A[p][s], make_uint4(o[0], o[1], o[2], o[3]), s == 0 ? O[p] : D[p][q]);
        }
      // under them: the previous stage's sums, and a quarter of the next unit's words
      const int pr = (rt + kGmRT - 1) % kGmRT, ps = rt == 0 ? up ^ 1 : up;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) y[pr][q][jj] += sc[ps][q] * D[p ^ 1][q][jj];
      if (rt == 0) scales(up ^ 1, sr[(u + 1) % kUnits]);
#pragma unroll
      for (int i = 0; i < kWords / kGmRT; ++i) {
        const int wi = rt * (kWords / kGmRT) + i;
        unpack(up ^ 1, wi, word(((u + 1) % kUnits) * KPG + wi / 4, wi % 4));
      }
      if (rt == kGmRT - 1) {
        // unit u + 1's words and scales are used: load those one chunk on
        const int un = (u + 1) % kUnits, cn = c + (u + 1) / kUnits + 1;
#pragma unroll
        for (int j = 0; j < KPG; ++j) wr[un * KPG + j] = wload(cn * kGmChunk + un * KPG + j);
        sr[un] = sload(cn * kUnits + un);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, KPG + (F16 ? 0 : 1), 0);  // the next stage's LDS reads
#pragma unroll
      for (int i = 0; i < 4 * KPG; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);            // one product
        __builtin_amdgcn_sched_group_barrier(0x002, KPG == 2 ? 4 : 6, 0);  // VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
      y[kGmRT - 1][q][jj] += sc[(kUnits - 1) & 1][q] * D[(kStages - 1) & 1][q][jj];

  if constexpr (GATED) {
    // gate | up sums meet in the chunk buffers, rounded to bf16 as the
    // projections' outputs are
    static_assert(sizeof(xs) >= (size_t)kGmRows * kGmCols * 2, "gate | up tile in the chunk buffers");
    uint16_t* yb = (uint16_t*)xs;
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < kGmRT; ++rt)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
        *(uint2*)(yb + (16 * rt + 4 * lq + jj) * kGmCols + 64 * wave + 4 * lr) =
            make_uint2(pack_bf16x2(y[rt][0][jj], y[rt][1][jj]), pack_bf16x2(y[rt][2][jj], y[rt][3][jj]));
    __syncthreads();
    const int c0 = ct * (kGmCols / 2);
    for (int i = tid; i < kGmRows * (kGmCols / 8); i += kGmThreads) {
      const int r = i / (kGmCols / 8), c = 4 * (i - r * (kGmCols / 8));
      const int row = rb * kGmRows + r;
      if (row >= a.M || c0 + c >= a.seg[0].N) continue;
      const uint2 g = *(const uint2*)(yb + r * kGmCols + c), v = *(const uint2*)(yb + r * kGmCols + kGmCols / 2 + c);
      const float h0 = round_to_bf16(gelu_tanh(bf16lo(g.x))) * bf16lo(v.x);
      const float h1 = round_to_bf16(gelu_tanh(bf16hi(g.x))) * bf16hi(v.x);
      const float h2 = round_to_bf16(gelu_tanh(bf16lo(g.y))) * bf16lo(v.y);
      const float h3 = round_to_bf16(gelu_tanh(bf16hi(g.y))) * bf16hi(v.y);
      gm_store4(a.seg[0].C + (size_t)row * a.seg[0].N + c0 + c, make_uint2(pack_bf16x2(h0, h1), pack_bf16x2(h2, h3)),
                a.c8);
    }
  } else {
    if (a.cap > 0.f) {
#pragma unroll
      for (int rt = 0; rt < kGmRT; ++rt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) y[rt][q][jj] = a.cap * tanhf(y[rt][q][jj] / a.cap);
    }
    const int row0 = rb * kGmRows + 4 * lq;
    uint16_t* cp = sg.C + (size_t)row0 * sg.N + col;
    const bool cok = col < sg.N;
    auto result = [&](int rt, int jj) {
      uint32_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) h[q] = moe::f32_to_act<F16>(y[rt][q][jj]);
      return make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    };
    if (a.c8) {
#pragma unroll
      for (int rt = 0; rt < kGmRT; ++rt)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
          if (cok && row0 + 16 * rt + jj < a.M) *(uint2*)(cp + (size_t)(16 * rt + jj) * sg.N) = result(rt, jj);
    } else {
#pragma unroll
      for (int rt = 0; rt < kGmRT; ++rt)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
          if (cok && row0 + 16 * rt + jj < a.M) gm_store4(cp + (size_t)(16 * rt + jj) * sg.N, result(rt, jj), 0);
    }
  }
}

// ---------------------------------------------------------------------------
// Few row blocks: the grid of the kernel above would leave most of the chip
// idle, so a workgroup owns 64 columns (GATED: 32 gate columns and the same 32
// up columns) and 16 RT rows, its 4 waves split K, and K is split over
// workgroups too.  A wave's k range is read straight into registers, two units
// ahead: the words of its 64 columns, and the token rows themselves (put into
// the words' k order there; their offset is one more product per row tile and
// k block), so there is one launch and no barrier before the sums.  The waves'
// sums meet in LDS; with a K split the last slice of a tile to arrive adds the
// fp32 partials in slice order.
// ---------------------------------------------------------------------------
struct GsArgs {
  const uint16_t* A;
  float* part;  // [ks][tiles][rows][64] (ks > 1)
  int* ctr;     // [tiles] arrival counters, zero between launches (ks > 1)
  int M, K, gs, rb, ks, upw;  // rb row blocks; upw units of k per wave
  int c8;
  float cap;
  GemmSeg seg[kMaxGemmSegs];
};

template <int KPG, int RT, bool F16, bool GATED>
__global__ __launch_bounds__(kGmThreads, 2) void gemm_small_kernel(GsArgs a) {
  constexpr int kRows = 16 * RT, kC = 64, kOutC = GATED ? 32 : 64;
  constexpr int kAhead = 2;  // units in flight per wave
  constexpr uint32_t kOob = 0xFFFFFFF0u;
  __shared__ float red[4][kRows][kC];
  __shared__ int last;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, lr = lane & 15;
  const int tile = blockIdx.x, slice = blockIdx.y;
  int ct = tile / a.rb;
  const int rb = tile - ct * a.rb;
  GemmSeg sg = a.seg[0];
  if constexpr (!GATED) {
#pragma unroll
    for (int i = 1; i < kMaxGemmSegs; ++i)
      if (ct >= a.seg[i].tile0) sg = a.seg[i];
    ct -= sg.tile0;
  }
  // columns past N read the last four (their results are not stored)
  const int c0 = ct * kOutC;
  const int colr = min(c0 + (GATED ? 4 * (lr & 7) : 4 * lr), sg.N - 4);
  const int32_t* bp = sg.B + colr;
  const uint16_t* sp = sg.S + colr;
  int G = sg.G, Gmax = sg.G;  // groups of the lane's columns; of the tile's
  if constexpr (GATED) {
    Gmax = max(G, a.seg[1].G);
    if (lr >= 8) {
      bp = a.seg[1].B + colr;
      sp = a.seg[1].S + colr;
      G = a.seg[1].G;
    }
  }
  const int Kp = a.K >> 3, units = (a.K + 32 * KPG - 1) / (32 * KPG);
  const int u0 = (slice * 4 + wave) * a.upw, u1 = min(units, u0 + a.upw);
  const int upg = a.gs / (32 * KPG);  // units per scale group
  const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(a.A, (uint32_t)a.M * (uint32_t)a.K * 2u);
  uint32_t roff[RT];  // rows past M read the last one (their results are not stored)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) roff[rt] = (uint32_t)min(rb * kRows + 16 * rt + lr, a.M - 1) * (uint32_t)a.K * 2u;

  // a unit past the wave's range, and a group past the scales, adds nothing:
  // its token rows read zeros and its scales count as zero.  The token rows
  // serve every lane's columns, so they end where the longer of two unequal
  // scale tables does; the shorter one's columns end by their scales (there a
  // non-finite value of the row is in the other factor of the result anyway).
  const int kend = min(min(a.K, 32 * KPG * u1), Gmax * a.gs);
  const int cend = min(kend, G * a.gs);
  u32x4_t xr[kAhead][RT][KPG], wr[kAhead][KPG];
  u32x2_t sr[kAhead];
  auto load = [&](int p, int u) {
#pragma unroll
    for (int s = 0; s < KPG; ++s) {
      const int kb = u * KPG + s, k = 32 * kb + 8 * lq;
      wr[p][s] = *(const u32x4_t*)(bp + (size_t)min(4 * kb + lq, Kp - 1) * sg.N);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        xr[p][rt][s] = __builtin_amdgcn_raw_buffer_load_b128(ra, k < kend ? roff[rt] + (uint32_t)k * 2u : kOob, 0, 0);
    }
    sr[p] = *(const u32x2_t*)(sp + (size_t)min(u / upg, G - 1) * sg.N);
  };
  const uint32_t mq = moe::q4_magic_t<F16>();
  const f32x4_t zf = {0.f, 0.f, 0.f, 0.f};
  const uint4 bc = make_uint4(moe::kQ4BiasPair, moe::kQ4BiasPair, moe::kQ4BiasPair, moe::kQ4BiasPair);
  f32x4_t y[RT][4];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int q = 0; q < 4; ++q) y[rt][q] = zf;
#pragma unroll
  for (int p = 0; p < kAhead; ++p) {
    load(p, u0 + p);
    __builtin_amdgcn_sched_barrier(0);  // (in the loop's order: its waits count the loads in between)
  }
#pragma unroll 1
  for (int ub = u0; ub < u1; ub += kAhead) {
#pragma unroll
    for (int p = 0; p < kAhead; ++p) {
      const int u = ub + p;
      uint4 B[KPG][4];
#pragma unroll
      for (int s = 0; s < KPG; ++s) {
        B[s][0] = moe::q4_operand_t<F16>(wr[p][s].x, mq);
        B[s][1] = moe::q4_operand_t<F16>(wr[p][s].y, mq);
        B[s][2] = moe::q4_operand_t<F16>(wr[p][s].z, mq);
        B[s][3] = moe::q4_operand_t<F16>(wr[p][s].w, mq);
#pragma unroll
        for (int q = 0; q < 4; ++q) B[s][q] = opaque(B[s][q]);  // unpacked here: the words' registers are free again
      }
      const bool live = 32 * KPG * u < cend;
      float sc[4] = {live ? moe::sc_lo<F16>(sr[p].x) : 0.f, live ? moe::sc_hi<F16>(sr[p].x) : 0.f,
                     live ? moe::sc_lo<F16>(sr[p].y) : 0.f, live ? moe::sc_hi<F16>(sr[p].y) : 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(sc[q]));
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        uint4 A[KPG];
        f32x4_t o = zf, D[4];
#pragma unroll
        for (int s = 0; s < KPG; ++s) {
          const u32x4_t v = xr[p][rt][s];
          A[s] = moe::mfma_k_order(make_uint4(v.x, v.y, v.z, v.w));
          if constexpr (!F16) o = moe::mfma_bf16(A[s], bc, o);
        }
#pragma unroll
        for (int s = 0; s < KPG; ++s)
#pragma unroll
          for (int q = 0; q < 4; ++q) D[q] = moe::mfma_act<F16>(A[s], B[s][q], s == 0 ? o : D[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) y[rt][q][jj] += sc[q] * D[q][jj];
      }
      __builtin_amdgcn_sched_barrier(0);
      load(p, u + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
      *(float4*)&red[wave][16 * rt + 4 * lq + jj][4 * lr] = make_float4(y[rt][0][jj], y[rt][1][jj], y[rt][2][jj], y[rt][3][jj]);
  __syncthreads();
  // a thread's results: 4 columns of a row (GATED: 4 gate columns and the same
  // up columns)
  constexpr int kQuads = kOutC / 4;
  auto finish = [&](int r, int c, float4 g, float4 v) {
    const int row = rb * kRows + r;
    if (row >= a.M || c0 + c >= sg.N) return;
    uint32_t h[4];
    const float gv[4] = {g.x, g.y, g.z, g.w}, vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float o = gv[q];
      if constexpr (GATED) o = round_to_bf16(gelu_tanh(round_to_bf16(o))) * round_to_bf16(vv[q]);
      else if (a.cap > 0.f) o = a.cap * tanhf(o / a.cap);
      h[q] = moe::f32_to_act<F16>(o);
    }
    gm_store4(sg.C + (size_t)row * sg.N + c0 + c, make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16)), a.c8);
  };
  auto add4 = [](float4 p, float4 q) { return make_float4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w); };
  auto wsum = [&](int r, int c) {
    return add4(add4(*(const float4*)&red[0][r][c], *(const float4*)&red[1][r][c]),
                add4(*(const float4*)&red[2][r][c], *(const float4*)&red[3][r][c]));
  };
  if (a.ks == 1) {
    for (int i = tid; i < kRows * kQuads; i += kGmThreads) {
      const int r = i / kQuads, c = 4 * (i - r * kQuads);
      finish(r, c, wsum(r, c), GATED ? wsum(r, c + 32) : make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }
  constexpr uint32_t kTileBytes = (uint32_t)kRows * kC * 4u;
  const size_t tiles = gridDim.x;
  const __amdgpu_buffer_rsrc_t rp = buffer_rsrc((char*)a.part + (slice * tiles + tile) * kTileBytes, kTileBytes);
  for (int i = tid; i < kRows * 16; i += kGmThreads) st_coherent_f4(rp, (uint32_t)i * 16u, wsum(i >> 4, 4 * (i & 15)));
  wait_vmem();
  __syncthreads();
  if (tid == 0) last = atomic_add_relaxed(&a.ctr[tile], 1) == a.ks - 1;
  __syncthreads();
  if (!last) return;
  // every slice's loads of a quad go out before they are added
  constexpr int kSlices = 16;
  auto psum = [&](int r, int c) {
    float4 v[kSlices];
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
      const __amdgpu_buffer_rsrc_t q =
          buffer_rsrc((char*)a.part + ((s < a.ks ? s : 0) * tiles + tile) * kTileBytes, s < a.ks ? kTileBytes : 0u);
      v[s] = ld_coherent_f4(q, (uint32_t)(r * 16 + (c >> 2)) * 16u);
    }
    float4 t = v[0];
#pragma unroll
    for (int s = 1; s < kSlices; ++s) t = add4(t, v[s]);  // slices past ks: zeros
    return t;
  };
  for (int i = tid; i < kRows * kQuads; i += kGmThreads) {
    const int r = i / kQuads, c = 4 * (i - r * kQuads);
    finish(r, c, psum(r, c), GATED ? psum(r, c + 32) : make_float4(0.f, 0.f, 0.f, 0.f));
  }
  if (tid == 0) store_relaxed(&a.ctr[tile], 0);
}

constexpr size_t kGmAlign = 256;
inline size_t gm_round(size_t v) { return (v + kGmAlign - 1) / kGmAlign * kGmAlign; }

// k blocks per unit: the largest of 2 and 1 whose width divides the group
int gm_kpg(int gs) { return gs % 64 == 0 ? 2 : 1; }

struct GmLayout {
  int KBp, Mp, units;
  size_t xf, off, total;
};
GmLayout gm_layout(int M, int K, int gs) {
  GmLayout l;
  l.KBp = ((K + 31) / 32 + kGmChunk - 1) / kGmChunk * kGmChunk;
  l.Mp = (M + kGmRows - 1) / kGmRows * kGmRows;
  l.units = l.KBp / gm_kpg(gs);
  l.xf = kGemmWsOffset;
  l.off = gm_round(l.xf + (size_t)l.Mp * l.KBp * 32 * 2);
  l.total = gm_round(l.off + (size_t)l.units * l.Mp * sizeof(float));
  return l;
}

template <int KPG, bool F16>
int launch_gm(const GmOrderArgs& o, const GmArgs& k, bool gated, hipStream_t stream) {
  hipLaunchKernelGGL((gemm_order_kernel<KPG, F16>), dim3((o.units + 3) / 4, k.rb * kGmRT), dim3(256), 0, stream, o);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "w4a16 gemm order launch");
  const dim3 grid(k.total), block(kGmThreads);
  if (!gated) hipLaunchKernelGGL((gemm_kernel<KPG, F16, false>), grid, block, 0, stream, k);
  else if constexpr (!F16) hipLaunchKernelGGL((gemm_kernel<KPG, false, true>), grid, block, 0, stream, k);
  else return fail(GI_ERR_UNSUPPORTED, "w4a16 gemm: the gated form takes bf16 rows");
  e = hipGetLastError();
  return e == hipSuccess ? GI_OK : hip_fail(e, "w4a16 gemm launch");
}

// The plan of a call: the large kernel, or the small one with ks K slices.
struct GmPlan {
  bool small;
  int rt, rb, tiles, ks, upw;  // small: row tiles per workgroup, row blocks, column tiles * rb, K slices, units per wave
  size_t bytes;
};
// From this many 64 x 256 workgroups on the large kernel is the faster one (K
// 2816-8192, whole calls, us, small / large: 128 of them 29.3 / 38.0 and 29.5 /
// 36.2, 88 of them 67.7 / 81.7; 176 of them 52.6 / 49.9 and 97.8 / 85.2; 256 of
// them 53.1 / 41.3).
constexpr int kGmMinWgs = 160;
constexpr int kGsTargetWgs = 256;
constexpr int kGsMaxSlices = 16;
constexpr int kGsMaxTiles = (int)(kGemmWsOffset / sizeof(int));

int gm_tiles(const int* N, int n, bool gated, int cols) {
  if (gated) return (N[0] + cols / 2 - 1) / (cols / 2);
  int t = 0;
  for (int i = 0; i < n; ++i) t += (N[i] + cols - 1) / cols;
  return t;
}

GmPlan gm_plan(int M, int K, int gs, const int* N, int n, bool gated) {
  GmPlan p{};
  const int kpg = gm_kpg(gs), units = (K + 32 * kpg - 1) / (32 * kpg);
  const GmLayout l = gm_layout(M, K, gs);
  p.rt = M <= 32 ? 2 : 4;
  p.rb = (M + 16 * p.rt - 1) / (16 * p.rt);
  p.tiles = gm_tiles(N, n, gated, 64) * p.rb;
  const long large = (long)gm_tiles(N, n, gated, kGmCols) * (l.Mp / kGmRows);
  p.small = large < kGmMinWgs && (long long)M * K * 2 < (1LL << 31);
  if (!p.small) {
    p.bytes = l.total;
    return p;
  }
  int ks = (kGsTargetWgs + p.tiles - 1) / p.tiles;
  if (ks > kGsMaxSlices) ks = kGsMaxSlices;
  if (p.tiles > kGsMaxTiles) ks = 1;
  p.upw = (units + 4 * ks - 1) / (4 * ks);
  p.ks = (units + 4 * p.upw - 1) / (4 * p.upw);
  p.bytes = p.ks > 1 ? gm_round(kGemmWsOffset + (size_t)p.ks * p.tiles * 16 * p.rt * 64 * sizeof(float)) : 0;
  return p;
}

template <int KPG, int RT, bool F16>
int launch_gs(const GsArgs& k, int tiles, bool gated, hipStream_t stream) {
  const dim3 grid(tiles, k.ks), block(kGmThreads);
  if (!gated) hipLaunchKernelGGL((gemm_small_kernel<KPG, RT, F16, false>), grid, block, 0, stream, k);
  else if constexpr (!F16) hipLaunchKernelGGL((gemm_small_kernel<KPG, RT, false, true>), grid, block, 0, stream, k);
  else return fail(GI_ERR_UNSUPPORTED, "w4a16 gemm: the gated form takes bf16 rows");
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GI_OK : hip_fail(e, "w4a16 gemm launch");
}
template <int KPG, bool F16>
int launch_gs_rt(const GsArgs& k, const GmPlan& p, bool gated, hipStream_t stream) {
  if (p.rt == 2) return launch_gs<KPG, 2, F16>(k, p.tiles, gated, stream);
  return launch_gs<KPG, 4, F16>(k, p.tiles, gated, stream);
}

int launch_small(const void* A, bool f16, int M, int K, int gs, float cap, const GemmSeg* segs, int nseg, bool gated,
                 const GmPlan& p, void* workspace, hipStream_t stream) {
  GsArgs k{};
  k.A = (const uint16_t*)A;
  k.M = M;
  k.K = K;
  k.gs = gs;
  k.rb = p.rb;
  k.ks = p.ks;
  k.upw = p.upw;
  k.cap = cap;
  k.c8 = 1;
  if (p.ks > 1) {
    k.ctr = (int*)workspace;
    k.part = (float*)((char*)workspace + kGemmWsOffset);
  }
  int tiles = 0;
  for (int i = 0; i < kMaxGemmSegs; ++i) {
    k.seg[i] = segs[i < nseg ? i : 0];
    k.seg[i].tile0 = i >= nseg ? 0x7fffffff : gated ? 0 : tiles;
    if (i < nseg && !gated) tiles += (segs[i].N + 63) / 64;
    if ((uintptr_t)k.seg[i].C % 8) k.c8 = 0;
  }
  if (gm_kpg(gs) == 2) return f16 ? launch_gs_rt<2, true>(k, p, gated, stream) : launch_gs_rt<2, false>(k, p, gated, stream);
  return f16 ? launch_gs_rt<1, true>(k, p, gated, stream) : launch_gs_rt<1, false>(k, p, gated, stream);
}

}  // namespace

bool gemm_supported(int M, int K, int gs, const int* N, int n) {
  if (M <= kGemmMinRows || gs <= 0 || gs % 32 || K <= 0 || K % 8 || n <= 0 || n > kMaxGemmSegs) return false;
  const GmLayout l = gm_layout(M, K, gs);
  long long tiles = 0;
  for (int i = 0; i < n; ++i) {
    // 32-bit offsets into the words (the chunks past K included) and scales
    if (N[i] < 4 || N[i] % 4 || (long long)(l.KBp + kGmChunk) * 4 * N[i] * 4 >= (1LL << 32)) return false;
    if ((long long)((K + gs - 1) / gs) * N[i] * 2 >= (1LL << 32)) return false;
    tiles += (N[i] + kGmCols / 2 - 1) / (kGmCols / 2);
  }
  return tiles * (l.Mp / kGmRows) < (1LL << 31) && l.Mp / 16 <= 65535;
}

size_t gemm_workspace_bytes(int M, int K, int gs, const int* N, int n, bool gated) {
  return gm_plan(M, K, gs, N, n, gated).bytes;
}

// An upper bound of gemm_workspace_bytes over every row count up to M that
// does not shrink as M grows (a plan's own need does: more rows need fewer K
// slices, and the large kernel needs other buffers).  The small kernel splits
// K only below kGsTargetWgs tiles, into ks <= kGsMaxSlices slices of ks * tiles
// < kGsTargetWgs + tiles tiles; the large kernel's buffers grow with M.
size_t gemm_workspace_bound(int M, int K, int gs, const int* N, int n, bool gated) {
  const GmPlan p = gm_plan(M, K, gs, N, n, gated);
  const size_t rows = M <= 32 ? 32 : 64;
  size_t b = p.small ? 0 : p.bytes;
  if (gm_tiles(N, n, gated, 64) < kGsTargetWgs) {
    size_t tiles = p.tiles < kGsTargetWgs ? p.tiles : kGsTargetWgs - 1;
    size_t slots = tiles + kGsTargetWgs - 1;
    if (slots > tiles * kGsMaxSlices) slots = tiles * kGsMaxSlices;
    const size_t s = gm_round(kGemmWsOffset + slots * rows * 64 * sizeof(float));
    if (s > b) b = s;
  }
  return b;
}

// given: the projections (gated: gate then up, the same N, out in given[0].C);
// the caller checked gemm_supported, the tensors and the workspace's size.
int launch_gemm(const void* A, bool f16, int M, int K, int gs, float cap, const GemmSeg* given, int nseg, bool gated,
                void* workspace, hipStream_t stream) {
  int N[kMaxGemmSegs];
  GemmSeg segs[kMaxGemmSegs];
  for (int i = 0; i < nseg; ++i) {
    segs[i] = given[i];
    segs[i].G = min(given[i].G, (K + gs - 1) / gs);  // groups past K are never read: 32-bit sizes and offsets hold
    N[i] = segs[i].N;
  }
  const GmPlan p = gm_plan(M, K, gs, N, nseg, gated);
  if (p.small) return launch_small(A, f16, M, K, gs, cap, segs, nseg, gated, p, workspace, stream);
  const GmLayout l = gm_layout(M, K, gs);
  GmOrderArgs o{};
  o.A = (const uint16_t*)A;
  o.xf = (uint4*)((char*)workspace + l.xf);
  o.off = (float*)((char*)workspace + l.off);
  o.M = M;
  o.K = K;
  o.KBp = l.KBp;
  o.units = l.units;
  GmArgs k{};
  k.xf = o.xf;
  k.off = o.off;
  k.M = M;
  k.K = K;
  k.KBp = l.KBp;
  k.gs = gs;
  k.rb = l.Mp / kGmRows;
  k.cap = cap;
  k.c8 = 1;
  int tiles = 0;
  for (int i = 0; i < kMaxGemmSegs; ++i) {
    if (i < nseg) {
      if ((uintptr_t)segs[i].C % 8) k.c8 = 0;
      k.seg[i] = segs[i];
      k.seg[i].tile0 = gated ? 0 : tiles;
      if (!gated) tiles += (segs[i].N + kGmCols - 1) / kGmCols;
    } else {
      k.seg[i] = segs[0];
      k.seg[i].tile0 = 0x7fffffff;
    }
  }
  if (gated) tiles = (segs[0].N + kGmCols / 2 - 1) / (kGmCols / 2);
  k.total = tiles * k.rb;
  if (gm_kpg(gs) == 2) return f16 ? launch_gm<2, true>(o, k, gated, stream) : launch_gm<2, false>(o, k, gated, stream);
  return f16 ? launch_gm<1, true>(o, k, gated, stream) : launch_gm<1, false>(o, k, gated, stream);
}

}  // namespace gi
