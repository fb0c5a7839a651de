// moe_midstream.hip -- grouped MXFP4 expert products for a few tokens per
// expert, on the gfx950 matrix cores.
//
// The same operation as grouped_mfma_kernel (moe_prefill.hip): for every
// expert of the routing plan, y = x W_e^T + b_e over the expert's rows, gated:
// bf16 gate/up and the clamped SwiGLU in the epilogue.  With tens of rows per
// expert the product is bound by the one read of the weights, so this kernel
// is a weight stream like the decode kernel's, with the tokens in LDS:
//
// * An item is (chunk of up to 64 rows of one expert) x (four 64-row weight
//   tiles); a work-group of four waves, a tile each, takes one item of every
//   round of G (grouped by XCD, so an XCD's work-groups share an expert's
//   token rows in L2).  Two work-groups run per CU (registers and LDS).
// * Each wave streams its tile's 1 KiB blocks with 16-byte nontemporal loads
//   into a ring of PB register slots: consuming block i of a phase (PB
//   blocks) issues block i of the next phase, which at the item's end is the
//   next item's first, so the stream does not stop between items.
// * The chunk's tokens of a phase sit in one of two LDS buffers.  Wave w loads
//   rows 16 w .. 16 w + 15 of a phase into registers one phase ahead and
//   writes them to LDS late in the phase before, so the waves synchronise
//   once per phase.  Rows past the chunk's end and blocks past K read past
//   the buffers: zeros, no traffic.
// * The next block's LDS reads and decode are placed between the products of
//   the current one; fragments of 16 rows past the second are multiplied only
//   where they hold rows.
//
// Numerics: one accumulator chain per output over the K blocks in order, the
// same instruction and order as grouped_mfma_kernel, so both give the same
// bits.
//
// Measured (GPT-OSS-120B layer, kernel trace, 200 tokens, uniform routing):
// gate_up 190 us against 227 in grouped_mfma_kernel, down 98 against 119; it
// reads 1.01 of the touched weights' bytes, at 6.0 TB/s.  What bounds it: a copy
// of the kernel without products and decode takes 184 us where this takes 200
// (450 tokens: 203 of 214), one without weight loads 165 (172), so neither the
// stream nor the rest hides wholly behind the other.  Waves issue for 0.49 of
// their cycles, wait to issue for 0.33 and on counters for 0.18; the matrix
// cores are busy for 0.3.
#include "moe_device.h"
#include "moe_kernels.h"

namespace gxmoe {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMidWaves = 4;              // waves per work-group, a 64-row weight tile each
constexpr int kMidPerCU = 2;              // work-groups per CU
constexpr int kMidFrags = 4;              // 16-row token fragments per chunk
constexpr int kMidRows = 16 * kMidFrags;  // rows per chunk
constexpr int kMidMaxRows = 1800;         // rows of a call (the rule by size, below)
constexpr int kMidChunks = kMaxExperts + kMidMaxRows / kMidRows;  // chunk table entries (LDS): all a call can have
constexpr int kBufWord3 = 0x00020000;     // raw buffer, dword data (gfx9 descriptor word 3)
constexpr int kNT = 2;                    // buffer load cache policy: nontemporal (streamed once)

struct MidParams {
  const uint16_t* x;         // [x_rows][K] bf16 rows
  const int32_t* row_index;  // [rows] permuted position -> row of x, or null (identity)
  const int32_t* offsets;    // [E+1] first permuted position of each expert
  const uint8_t* wn;         // tiled nibbles, g.nib_bytes per expert
  const uint8_t* ws;         // tiled scales, g.scale_bytes per expert
  const uint16_t* bias;      // [E][N] or null
  uint16_t* out;             // gated: [rows][N/2] activations; else [rows][N]
  uint16_t* gate_up;         // gated and optional: [rows][N] bf16 gate/up values
  uint32_t x_bytes, idx_bytes, wn_bytes, ws_bytes, bias_bytes, out_bytes;  // buffer extents (each < 2^32 - 2^16)
  int E, num_cus;
  float alpha, limit;
  TiledGeom g;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), kBufWord3);
}

__device__ __forceinline__ bool any_special(const gx_u32x4& v) {
  return has_special_code(v[0], 0xffffffffu) | has_special_code(v[1], 0xffffffffu) |
         has_special_code(v[2], 0xffffffffu) | has_special_code(v[3], 0xffffffffu);
}

// One item, wave-uniform.  A missing item has no rows and every load past its
// buffer's end.
struct MidItem {
  int valid, e, p0, mc, tile;  // expert, first permuted row, rows, this wave's weight tile
};

template <bool kGated, int PB>
__global__ __launch_bounds__(kMidWaves * kWave, kMidPerCU) void mid_stream_kernel(MidParams a) {
  constexpr int NC = kMidFrags;
  constexpr int kBuf = PB * NC * 1024;   // bytes of a phase's tokens: KiB (block i, fragment t) at (NC i + t)
  constexpr int kIssue = 3;                          // tokens written and loaded per block
  constexpr int kLead = (PB + kIssue - 1) / kIssue;  // over this many blocks ahead of the last
  static_assert(kMidWaves == NC && kLead + 2 < PB, "wave w stages fragment w");
  __shared__ __attribute__((aligned(1024))) uint8_t xs[2 * kBuf];
  // each wave's scales of a phase and its bias rows; the lanes past them write
  // the element after the end (no branch in the block loop)
  __shared__ gx_u32x4 scs[kMidWaves][2][PB * 4 + 1];
  __shared__ uint2 bs[kMidWaves][kTileRows / 4 + 1];
  __shared__ int2 tab[kMidChunks];                // chunks: {expert | rows << 8, first permuted row}
  __shared__ int tab_n, tail_item;

  static_assert((sizeof(xs) + sizeof(scs) + sizeof(bs) + sizeof(tab) + sizeof(tab_n) + sizeof(tail_item)) * kMidPerCU <=
                    160 * 1024,
                "two work-groups per CU");

  const TiledGeom& g = a.g;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int K = g.K, N = g.N, nb = g.nb;
  const int ntiles = N / kTileRows, ngrp = (ntiles + kMidWaves - 1) / kMidWaves;
  const int nph = (nb + PB - 1) / PB;

  // The chunk table from the plan's offsets: lane l holds experts 4 l .. 4 l + 3.
  if (w == 0) {
    constexpr int kPer = kMaxExperts / kWave;
    int o[kPer + 1], n = 0;
#pragma unroll
    for (int i = 0; i <= kPer; ++i) o[i] = a.offsets[min(lane * kPer + i, a.E)];
#pragma unroll
    for (int i = 0; i < kPer; ++i) n += (o[i + 1] - o[i] + kMidRows - 1) / kMidRows;
    int s = n;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int t = __shfl_up(s, d, kWave);
      if (lane >= d) s += t;
    }
    if (lane == kWave - 1) tab_n = s;
    s -= n;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      for (int p = o[i]; p < o[i + 1]; p += kMidRows)
        if (s < kMidChunks) tab[s++] = make_int2((lane * kPer + i) | (min(kMidRows, o[i + 1] - p) << 8), p);
  }
  __syncthreads();
  const int n_items = min(__builtin_amdgcn_readfirstlane(tab_n), kMidChunks) * ngrp;
  // Items go in rounds of G, XCD b % 8 taking consecutive ones.  A last round
  // of at most one item per CU is dealt evenly to the XCDs: packed into the
  // first of them, 92 items (200 rows on four experts) ran on two XCDs in
  // 48 us, spread over eight in 33, and the 128 left of 1664 (200 rows on 128
  // experts) cost 157 us against 138.  A fuller one stays packed: it puts two
  // work-groups on most CUs either way (2944 items: 193 us, spread 194).
  const int G = gridDim.x;  // a multiple of 8
  const int full = n_items / G * G;  // items of the full rounds
  int q;                             // this work-group's item, -1: none
  {
    const int xcd = static_cast<int>(blockIdx.x) & 7, slot = static_cast<int>(blockIdx.x) >> 3;
    const int left = n_items - full;
    const int share = left > a.num_cus ? G >> 3 : (left + 7) >> 3;
    const int o = xcd * share + slot;
    const int tail = slot < share && o < left ? full + o : -1;
    if (threadIdx.x == 0) tail_item = tail;
    q = full > 0 ? xcd * (G >> 3) + slot : tail;
  }
  if (q < 0) return;
  auto next_item = [&]() -> int {
    return q + G < full ? q + G : q < full ? __builtin_amdgcn_readfirstlane(tail_item) : -1;
  };

  const __amdgpu_buffer_rsrc_t rX = rsrc_of(a.x, a.x_bytes);
  const __amdgpu_buffer_rsrc_t rI = rsrc_of(a.row_index, a.idx_bytes);
  const __amdgpu_buffer_rsrc_t rA = rsrc_of(a.wn, a.wn_bytes);
  const __amdgpu_buffer_rsrc_t rS = rsrc_of(a.ws, a.ws_bytes);
  const __amdgpu_buffer_rsrc_t rB = rsrc_of(a.bias, a.bias_bytes);
  const __amdgpu_buffer_rsrc_t rO = rsrc_of(a.out, a.out_bytes);

  auto item_of = [&](int qq) -> MidItem {
    MidItem s;
    s.valid = qq >= 0;
    const int j = s.valid ? qq / ngrp : 0;
    s.tile = (qq - j * ngrp) * kMidWaves + w;
    const int hx = __builtin_amdgcn_readfirstlane(tab[j].x);
    s.e = hx & 0xff;
    s.mc = s.valid ? hx >> 8 : 0;
    s.p0 = __builtin_amdgcn_readfirstlane(tab[j].y);
    return s;
  };
  // Byte offsets of an item's first weight block and scale group; a wave past
  // the last tile (or a missing item) reads past the end.
  auto live = [&](const MidItem& s) { return s.valid && s.tile < ntiles; };
  auto a_of = [&](const MidItem& s) -> uint32_t {
    return static_cast<uint32_t>(s.e) * static_cast<uint32_t>(g.nib_bytes) + static_cast<uint32_t>(s.tile * nb) * 1024u;
  };
  auto s_of = [&](const MidItem& s) -> uint32_t {
    return static_cast<uint32_t>(s.e) * static_cast<uint32_t>(g.scale_bytes) + static_cast<uint32_t>(g.mscale_off) +
           static_cast<uint32_t>(s.tile * nb) * 64u;
  };

  // Token staging: this lane moves 16 bytes (quarter lane % 4) of row
  // lane / 4 of fragment w per block.  LDS unit 4 j + (q ^ swz(j)) of a KiB holds
  // quarter q of its row j, swz(j) = (j / 2) % 4: the 16 rows read at one
  // quarter by a fragment load hit distinct banks.
  const int sj = lane >> 2, srow = 16 * w + sj;
  const int xw = 1024 * w + 64 * sj + 16 * ((lane & 3) ^ ((sj >> 1) & 3));
  const int bj = lane & 15;
  const int boff = bj * 64 + 16 * ((lane >> 4) ^ ((bj >> 1) & 3));
  auto xrow = [&](const MidItem& s, int row) -> uint32_t {  // row of x -> byte offset of this lane's piece
    return srow < s.mc ? static_cast<uint32_t>(row) * static_cast<uint32_t>(K) * 2u + 16u * (lane & 3) : a.x_bytes;
  };
  auto idx_off = [&](const MidItem& s) -> uint32_t {
    return srow < s.mc ? static_cast<uint32_t>(s.p0 + srow) * 4u : a.idx_bytes;
  };
  const bool gather = a.row_index != nullptr;
  // Scalar offset of K block b.  The range check compares the lane's offset
  // with the extent less the scalar offset, so the latter stays within the
  // extent: 0 for a block past K, which with one row of x would lie past it.
  auto xblk = [&](int b) -> int { return b < nb ? 64 * b : 0; };

  gx_u32x4 ra[PB];   // the weight ring: slot i = block i of the phase being (or next) consumed
  gx_u32x4 xt[PB];   // a phase's tokens on their way to LDS
  const uint32_t voffA = 16u * lane;
  bool spec = false;  // a scale of the item holds code 0 or 255
  int buf = 0;

  // First item: its first phase's operands, waited for.
  MidItem cur = item_of(q);
  uint32_t vx = 0;  // this lane's token row of the current item
  {
    const int row = gather && srow < cur.mc ? a.row_index[cur.p0 + srow] : cur.p0 + srow;
    vx = xrow(cur, row);
    const bool lv = live(cur);
    const uint32_t sa = a_of(cur), ss = s_of(cur);
#pragma unroll
    for (int r = 0; r < PB; ++r) xt[r] = __builtin_amdgcn_raw_buffer_load_b128(rX, vx, 64 * r, 0);
    const gx_u32x4 sv = __builtin_amdgcn_raw_buffer_load_b128(
        rS, lane < 4 * min(PB, nb) ? 16u * lane : a.ws_bytes, lv ? ss : a.ws_bytes, kNT);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      ra[i] = __builtin_amdgcn_raw_buffer_load_b128(rA, voffA, lv && i < nb ? sa + 1024u * i : a.wn_bytes, kNT);
#pragma unroll
    for (int r = 0; r < PB; ++r) *reinterpret_cast<gx_u32x4*>(xs + xw + 1024 * NC * r) = xt[r];
    // the second phase's tokens stay in flight: phase p writes phase p + 1's
#pragma unroll
    for (int r = 0; r < PB; ++r)
      xt[r] = __builtin_amdgcn_raw_buffer_load_b128(rX, PB + r < nb ? vx : a.x_bytes, xblk(PB + r), 0);
    scs[w][0][min(lane, 4 * PB)] = sv;
    spec = lv && lane < 4 * min(PB, nb) && any_special(sv);
  }
  lds_barrier();

  // Operands of the block about to be multiplied and the scale of the next.
  gx_bf16x8 av[4], bv[NC];
  uint32_t sc;
  auto decode = [&](const gx_u32x4& v, uint32_t c, gx_bf16x8 (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) o[s] = decode8_bf16(v[s], __uint_as_float(((c >> (8 * s)) & 0xffu) << 23));
  };
  {
    const uint32_t* const sr = reinterpret_cast<const uint32_t*>(scs[w][0]) + bj;
#pragma unroll
    for (int t = 0; t < NC; ++t) bv[t] = *reinterpret_cast<const gx_bf16x8*>(xs + boff + 1024 * t);
    sc = sr[16];
    decode(ra[0], sr[0], av);
  }

  for (;;) {
    q = next_item();
    const MidItem nxt = item_of(q);
    uint32_t vxn = 0;    // the next item's token row
    bool nspec = false;  // special codes seen in the next item's first phase
    {
      f32x4 acc[4][NC];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NC; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

      for (int ph = 0; ph < nph; ++ph) {
        // What this phase loads: the item's next phase, or the next item's first.
        const bool last = ph + 1 == nph;
        const bool lv = last ? live(nxt) : live(cur);
        const int b0 = last ? 0 : (ph + 1) * PB;  // its first block
        const int nlive = min(PB, nb - b0);       // its blocks below nb
        const uint32_t na = (last ? a_of(nxt) : a_of(cur)) + 1024u * b0;
        const uint32_t ns = lv ? (last ? s_of(nxt) : s_of(cur)) + 64u * b0 : a.ws_bytes;
        // Tokens are loaded a phase earlier than weights (written to LDS a
        // phase after their load): phase ph + 2, or the next item's ph + 2 - nph.
        const bool xnext = ph + 2 >= nph;
        const int xb0 = (xnext ? ph + 2 - nph : ph + 2) * PB;
        // fragments multiplied: the last block of the item reads the next
        // item's first fragments
        const int nfe = (max(cur.mc, last ? nxt.mc : 0) + 15) >> 4;
        // this phase's and the next phase's buffers
        const uint8_t* const xr = xs + buf * kBuf + boff;
        const uint8_t* const xrn = xs + (buf ^ 1) * kBuf + boff;
        uint8_t* const xwr = xs + (buf ^ 1) * kBuf + xw;
        const uint32_t* const sr = reinterpret_cast<const uint32_t*>(scs[w][buf]) + bj;
        const uint32_t* const srn = reinterpret_cast<const uint32_t*>(scs[w][buf ^ 1]) + bj;

        const gx_u32x4 sv =
            __builtin_amdgcn_raw_buffer_load_b128(rS, lane < 4 * nlive ? 16u * lane : a.ws_bytes, ns, kNT);
        const uint32_t rid = __builtin_amdgcn_raw_buffer_load_b32(rI, idx_off(nxt), 0, 0);
        const gx_u32x2 bv2 = __builtin_amdgcn_raw_buffer_load_b64(
            rB, live(cur) && lane < kTileRows / 4 ? (static_cast<uint32_t>(cur.e) * N + cur.tile * kTileRows) * 2u + 8u * lane
                                                  : a.bias_bytes, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // Block i's products run while block i + 1's token fragments are read
        // and its weights decoded.  A wave issues in order, so the reads and
        // the decode are placed between the products: behind them they would
        // leave the matrix core idle.  All reads of this phase's buffers
        // are issued by block PB - 2; the barrier ahead of the last block
        // then shows every wave's writes of the next phase.
#pragma unroll
        for (int i = 0; i < PB; ++i) {
          if (i == PB - 1) lds_barrier();
          if (i == PB - 1 - kLead) vxn = xrow(nxt, gather ? static_cast<int>(rid) : nxt.p0 + srow);
          gx_bf16x8 an[4], bn[NC];
          auto read_frag = [&](int t) __attribute__((always_inline)) {
            bn[t] = *reinterpret_cast<const gx_bf16x8*>(i + 1 < PB ? xr + 1024 * (NC * (i + 1) + t) : xrn + 1024 * t);
          };
          auto products = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
              acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s], bv[t], acc[s][t], 0, 0, 0);
          };
          const uint32_t scn = i + 2 < PB ? sr[16 * (i + 2)] : srn[16 * (i + 2 - PB)];
          read_frag(0);
          read_frag(1);
          ra[i] = __builtin_amdgcn_raw_buffer_load_b128(rA, voffA, lv && i < nlive ? na + 1024u * i : a.wn_bytes, kNT);
          products(0);
          products(1);
          decode(ra[(i + 1) % PB], sc, an);
          if (i >= PB - 1 - kLead && i < PB - 1) {
#pragma unroll
            for (int r = kIssue * (i - PB + 1 + kLead); r < kIssue * (i - PB + 2 + kLead) && r < PB; ++r) {
              *reinterpret_cast<gx_u32x4*>(xwr + 1024 * NC * r) = xt[r];
              xt[r] = __builtin_amdgcn_raw_buffer_load_b128(rX, xb0 + r < nb ? (xnext ? vxn : vx) : a.x_bytes,
                                                            xblk(xb0 + r), 0);
            }
          }
          if (i == PB - 3) {
            scs[w][buf ^ 1][min(lane, 4 * PB)] = sv;
            bs[w][min(lane, kTileRows / 4)] = make_uint2(bv2[0], bv2[1]);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // the scale
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
#pragma unroll
          for (int m = 2; m < 8; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (nfe > 2) {
            read_frag(2);
            products(2);
          }
          if (nfe > 3) {
            read_frag(3);
            products(3);
          }
#pragma unroll
          for (int s = 0; s < 4; ++s) av[s] = an[s];
#pragma unroll
          for (int t = 0; t < NC; ++t) bv[t] = bn[t];
          sc = scn;
          __builtin_amdgcn_sched_barrier(0);  // one block at a time: the ring's load order is the wait order
        }
        const bool sp = lv && lane < 4 * nlive && any_special(sv);
        if (last) nspec = sp;
        else spec = spec || sp;
        buf ^= 1;
      }

      if (live(cur)) {
      // Scale codes 0 and 255 (none in a regular checkpoint): the wave's tile
      // again, block by block, with the reference's decode of those codes.
      if (__builtin_expect(__ballot(spec) != 0ull, 0)) {
        uint32_t trow[NC];
#pragma unroll
        for (int t = 0; t < NC; ++t) {
          const int p = cur.p0 + min(16 * t + bj, cur.mc - 1);
          trow[t] = static_cast<uint32_t>(gather ? a.row_index[p] : p) * static_cast<uint32_t>(K) * 2u + 16u * (lane >> 4);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < NC; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int kb = 0; kb < nb; ++kb) {
          const gx_u32x4 wv = __builtin_amdgcn_raw_buffer_load_b128(rA, voffA, a_of(cur) + 1024u * kb, 0);
          const uint32_t sv = __builtin_amdgcn_raw_buffer_load_b32(rS, 4u * bj, s_of(cur) + 64u * kb, 0);
          gx_bf16x8 av[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) av[s] = decode8_bf16_special(wv[s], (sv >> (8 * s)) & 0xffu);
#pragma unroll
          for (int t = 0; t < NC; ++t) {
            const gx_bf16x8 b1 =
                __builtin_bit_cast(gx_bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rX, trow[t], 64 * kb, 0));
#pragma unroll
            for (int s = 0; s < 4; ++s)
              acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s], b1, acc[s][t], 0, 0, 0);
          }
        }
      }

      // Epilogue: acc[i][t][r] is row 16 i + 4 (lane / 16) + r of the tile for
      // token 16 t + lane % 16; rows past the chunk store past the buffer.
      const int n0 = cur.tile * kTileRows + 4 * (lane >> 4);
      uint2 bb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) bb[i] = bs[w][4 * i + (lane >> 4)];
#pragma unroll
      for (int t = 0; t < NC; ++t) {
        if (16 * t >= cur.mc) break;
        const int j = 16 * t + bj;
        const uint32_t p = static_cast<uint32_t>(cur.p0 + j);
        const uint32_t vo = j < cur.mc ? (kGated ? p * N + n0 : 2u * (p * N + n0)) : a.out_bytes;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t y01 = pack_bf16x2(acc[i][t][0] + __uint_as_float(bb[i].x << 16),
                                           acc[i][t][1] + __uint_as_float(bb[i].x & 0xffff0000u));
          const uint32_t y23 = pack_bf16x2(acc[i][t][2] + __uint_as_float(bb[i].y << 16),
                                           acc[i][t][3] + __uint_as_float(bb[i].y & 0xffff0000u));
          if constexpr (kGated) {
            // rows n, n+2 are gate (even), n+1, n+3 up (odd)
            const float a0 = gx_swiglu(__uint_as_float(y01 << 16), __uint_as_float(y01 & 0xffff0000u), a.alpha, a.limit);
            const float a1 = gx_swiglu(__uint_as_float(y23 << 16), __uint_as_float(y23 & 0xffff0000u), a.alpha, a.limit);
            __builtin_amdgcn_raw_buffer_store_b32(pack_bf16x2(a0, a1), rO, vo + 16u * i, 0, 0);
            if (a.gate_up && j < cur.mc)
              *reinterpret_cast<uint2*>(a.gate_up + static_cast<size_t>(p) * N + n0 + 16 * i) = make_uint2(y01, y23);
          } else {
            __builtin_amdgcn_raw_buffer_store_b64(gx_u32x2{y01, y23}, rO, vo + 32u * i, 0, 0);
          }
        }
      }
      }
    }
    if (!nxt.valid) break;
    cur = nxt;
    vx = vxn;
    spec = nspec;
  }
}

template <bool kGated, int PB>
hipError_t launch_mid_t(const MidParams& p, int grid, hipStream_t s, const KernelTimer& t) {
  gx_launch(mid_stream_kernel<kGated, PB>, dim3(grid), dim3(kMidWaves * kWave), 0, s, t, p);
  return hipGetLastError();
}

}  // namespace

// The rule by size.  Measured, GPT-OSS shapes, layer us (grouped_mfma_kernel /
// this kernel), uniform and Zipf(1.1) routing: 128 experts, 512 rows 356 / 296
// and 277 / 261; 800 rows 357 / 303 and 320 / 281; 2048 rows 396 / 342 and 392 /
// 393; 4004 rows 443 / 400 but 461 / 506: a few experts then hold most rows, and
// a 64-row chunk costs their products more than a 128-row tile does.  32
// experts, 800 rows 139 / 120 and 169 / 132; 1600 rows 163 / 155 and 191 / 170;
// 2400 rows 186 / 240.  So: up to 1800 rows, and up to 50 on average per expert.
//
// Over what the rule admits, one product at a time (1 to 256 experts, eight
// shapes from 64 x 320 to 5760 x 2880, 8 to 1800 rows, uniform and Zipf(1.1)
// routing and all rows on four experts or one; 2184 points), this kernel takes
// 0.75 of the other's time on average and at most 1.03, but for down products
// of 64 experts, 2880 x 2880, 800 to 1600 rows, where single Zipf draws reach
// 1.08 (0.97 over eight draws).  Closest: 1800 rows on one expert, gate_up of
// the 120B layer, 75.5 / 74.5 us.
bool mid_stream_pays(const GroupedArgs& a) {
  const int active = a.E < a.rows ? a.E : a.rows;
  return a.rows <= kMidMaxRows && a.rows <= 50 * active;
}

bool mid_stream_supported(const GroupedArgs& a) {
  if (!grouped_supported(a.N, a.K, a.E) || a.x_rows <= 0 || a.num_cus <= 0 || a.xq != nullptr) return false;
  const TiledGeom g = tiled_geom(a.N, a.K);
  if (g.nb <= 9) return false;  // one phase: a next item's rows would not be known in time
  if (a.rows > kMidMaxRows) return false;  // the chunk table
  constexpr size_t kMaxBuf = 0xffff0000u;  // 32-bit buffer offsets, with room for the lanes' terms
  const size_t S = static_cast<size_t>(a.rows);
  return g.nib_bytes * a.E <= kMaxBuf && g.scale_bytes * a.E <= kMaxBuf && S * 4 <= kMaxBuf &&
         static_cast<size_t>(a.x_rows) * a.K * 2 <= kMaxBuf && S * a.N * 2 <= kMaxBuf &&
         static_cast<size_t>(a.E) * a.N * 2 <= kMaxBuf;
}

hipError_t launch_mid_stream(const GroupedArgs& a, hipStream_t s) {
  if (a.rows <= 0) return hipSuccess;
  if (!mid_stream_supported(a)) return hipErrorInvalidValue;
  MidParams p{};
  p.x = a.x;
  p.row_index = a.row_index;
  p.offsets = a.offsets;
  p.wn = a.wn;
  p.ws = a.ws;
  p.bias = a.bias;
  p.out = a.out;
  p.gate_up = a.gated ? a.gate_up : nullptr;
  p.g = tiled_geom(a.N, a.K);
  p.x_bytes = static_cast<uint32_t>(static_cast<size_t>(a.x_rows) * a.K * 2);
  p.idx_bytes = a.row_index ? static_cast<uint32_t>(a.rows) * 4u : 0u;
  p.wn_bytes = static_cast<uint32_t>(p.g.nib_bytes * a.E);
  p.ws_bytes = static_cast<uint32_t>(p.g.scale_bytes * a.E);
  p.bias_bytes = a.bias ? static_cast<uint32_t>(static_cast<size_t>(a.E) * a.N * 2) : 0u;
  p.out_bytes = static_cast<uint32_t>(static_cast<size_t>(a.rows) * (a.gated ? a.N / 2 : a.N) * 2);
  p.E = a.E;
  p.num_cus = a.num_cus;
  p.alpha = a.alpha;
  p.limit = a.limit;
  const int ngrp = (a.N / kTileRows + kMidWaves - 1) / kMidWaves;
  const int active = a.E < a.rows ? a.E : a.rows;
  const long items = static_cast<long>(active + a.rows / kMidRows) * ngrp, slots = static_cast<long>(kMidPerCU) * a.num_cus;
  const int grid = static_cast<int>(((items < slots ? items : slots) + 7) & ~7L);
  // phases of 8 or 9 blocks: whichever leaves fewer past K (9 for K = 2880)
  const bool eight = (p.g.nb + 7) / 8 * 8 < (p.g.nb + 8) / 9 * 9;
  if (a.gated) return eight ? launch_mid_t<true, 8>(p, grid, s, a.timer) : launch_mid_t<true, 9>(p, grid, s, a.timer);
  return eight ? launch_mid_t<false, 8>(p, grid, s, a.timer) : launch_mid_t<false, 9>(p, grid, s, a.timer);
}

}  // namespace gxmoe
