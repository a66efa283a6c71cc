// Key split of attention over few query rows per KV head (decode, chain verification: up to 64 rows).
//
// The keys of a group (request, KV head) are cut into splits of 2048 to 8192 (split_log2()), a split's tiles are dealt
// round robin to four waves (with more than 32 rows, two pairs of waves), and a wave's tiles into units (unit_log2()).
// Each unit is walked with a state of its own; a wave's units are folded in order, the waves of a split are merged, the
// split is rounded to the partial type, and the splits are merged by weight.  This cut, and so a row's arithmetic, is a
// function of the group's own rows and length only (a request gives the same bits alone, in a batch and in a longer
// cache), while two kinds of launch evaluate it:
//   * key_split_kernel, one workgroup per split: the units are folded in the waves' registers;
//   * key_units_kernel, when there are too few splits for the chip (one request of 8192 keys: 32): the units are dealt
//     out to all waves and stored, and the combine launch folds them (key_units_combine_kernel).
// A stored unit is not free: its stores wait in the queue that the tile loads of a memory-bound launch fill (1.1 us a
// unit in decode, 3.1 us with 32 rows, against 2.4 us a tile, every wave at once), so launches that fill the chip
// store once per split.
#pragma once
#include "attn_core.h"
#include "vmk_internal.h"

namespace vmk {

struct KeySplitArgs {
  const f16* q;            // (B, kd, Hq, 128)
  const f16* k;            // (B, Hkv, L, 128); paged: the page pools, num_pages pages of ps rows, HND or NHD
  const f16* v;
  const uint32_t* bits;    // (B, kd, W), or null: every cache position visible to every query row (plain decode)
  const int* lens;         // (B,) cache positions in use per batch entry (clamped to [kd, L]), or null: all L
  const int* pages;        // paged: (B, max_pages) page table
  // Partials, [grp - g0][row block][slots][rows_s][128] and their (m, l) pairs: splits as normalised O rows of part_t,
  // or of fp32 where split_wide() (one row block), or units as fp32 sums (row blocks of 32 rows).
  void* part_o;
  float* part_ml;
  void* out;               // (B, kd, Hq, 128)
  int B, kd, Hq, Hkv, G, L, W;
  int ps, max_pages, num_pages;
  int esize;               // bytes that an element of a split's rows is given (fp16 rows fill half of 4)
  int nrb, slots, rows_s;  // row blocks of a group; splits or units per (group, row block), at most; rows of one partial
  int g0, ngrp;            // groups of this launch (with lens: all of them)
  int logw;                // units: log2 of the shares the line of tiles is cut into (four waves each)
  float sl2;               // softmax scale * log2(e)
};

// Waves that interleave a split's tiles.
__host__ __device__ inline int split_waves(int rows) { return rows <= 32 ? 4 : 2; }
__host__ __device__ inline int split_waves_log2(int rows) { return rows <= 32 ? 2 : 1; }

// log2 of the keys of a split, for a group of `rows` query rows whose own length is n: 2048 keys up to 28 rows (decode:
// 256 workgroups once B * Hkv * L reaches 2^19).  With more rows a split's partial is larger, and requests past 16384
// positions take 4096 (32 rows, four requests of 32768 keys: 94 us against 102 with 2048; 24 rows, one request of 50919
// keys: 55.2 us against 46.8); past a million positions every split of more than 16 rows does, and of more than 32 rows
// 8192, so that the partials of one group stay within the allocation-free scratch.  The steps are whole tiles, so n may
// be rounded up to its tiles.  Shifts: divisions made one request of 8 drafts over 8192 keys 0.25 us longer.
constexpr int kSplitStep1 = 16384, kSplitStep2 = 1 << 20;
template <class N>
__host__ __device__ inline int split_log2(int rows, N n) {
  if (rows <= 16 || n <= (rows <= 28 ? kSplitStep2 : kSplitStep1)) return 11;
  return rows > 32 && n > kSplitStep2 ? 13 : 12;
}
// Splits of a group of n positions.
template <class N>
__host__ __device__ inline N group_splits(int rows, N n) {
  const int s = split_log2(rows, n);
  return (n + (1 << s) - 1) >> s;
}

// Whether a group's splits stay fp32 for fp16 inputs: groups of more than 16 rows and of up to 128 keys per row, which
// 2048 keys cut into two to four.  As one split their rows would be rounded once, so rounding the splits would add an
// error that one split does not have (12 drafts over 5000 keys, relative error 2.92e-4 as one split, 3.53e-4 as three
// in fp16, 2.88e-4 in fp32).  Longer groups have several splits of either size and round them to fp16 as ever. The rows
// are twice the bytes: 16 drafts, 8 requests of 8192 keys 51.1 us for 51.0, 9 drafts of 5000 35.8 for 35.5, 16 drafts,
// 32 requests of 8192 keys 224 for 214.
template <class N>
__host__ __device__ inline bool split_wide(int rows, N n) {
  return rows > 16 && n > 2048 && n <= 128 * rows;
}

// log2 of the tiles of a unit of a group with nt key tiles: about 64 units to a group, at least four or eight tiles (a
// unit's partial is rows * 528 bytes, its keys 16 KB a tile), at most the wave's tiles of a split.
__host__ __device__ inline int unit_log2(int rows, int nt) {
  const int hi = split_log2(rows, nt * kTile) - 5 - split_waves_log2(rows);
  int t = rows <= 8 ? 2 : 3;
  while (t < hi && (64 << t) < nt) ++t;
  return t;
}
__host__ __device__ inline int unit_tiles(int rows, int nt) { return 1 << unit_log2(rows, nt); }
// Units of a group of nt tiles: blocks of split_waves() units, but for a last block of fewer tiles than that.
__host__ __device__ inline int group_units(int rows, int nt) {
  const int q = split_waves(rows), bt = unit_log2(rows, nt) + split_waves_log2(rows);   // tiles of a block, log2
  const int nb = (nt + (1 << bt) - 1) >> bt, last = nt - ((nb - 1) << bt);
  return (nb - 1) * q + (last < q ? last : q);
}
// The most splits, and the most units (up to 64 units of one size, then of the next; past 64 of the largest size, as
// many as there are), of a group of 1 .. L keys.  Both fall where the split size steps up, so the lengths at the steps
// count, too.
template <class F>
inline int64_t most_up_to(int64_t L, F f) {
  return std::max(f(L), std::max(f(std::min<int64_t>(L, kSplitStep1)), f(std::min<int64_t>(L, kSplitStep2))));
}
inline int64_t split_slots(int rows, int64_t L) {
  return most_up_to(L, [&](int64_t n) { return group_splits(rows, n); });
}
inline int64_t unit_slots(int rows, int64_t L) {
  return most_up_to(L, [&](int64_t n) {
    return std::max<int64_t>(std::min<int64_t>(64, (n + kTile - 1) / kTile), split_waves(rows) * group_splits(rows, n));
  });
}

// Cache positions of batch entry b: lens[b] clamped to [kd, L] (the query rows are the last kd of them), or L.
__device__ __forceinline__ int stream_len(const KeySplitArgs& a, int b) {
  return a.lens ? min(max(a.lens[b], a.kd), a.L) : a.L;
}
// The same for a wave-uniform b, as a scalar load (no wait on the vector-memory loads in flight).
__device__ __forceinline__ int stream_len_uniform(const KeySplitArgs& a, int b) {
  if (!a.lens) return a.L;
  const int n = *(const int __attribute__((address_space(4)))*)(const void __attribute__((address_space(4)))*)(a.lens + b);
  return min(max(n, a.kd), a.L);
}
__device__ __forceinline__ int tiles_of(int n) { return (n + kTile - 1) >> 5; }

// A block of split_waves() units' place: its group and first tile within the group; (the first group past the launch's,
// 0) is the end.
struct StreamPos {
  int g, t;
};

// The first block at or after tile t of group g (nt tiles).
__device__ __forceinline__ StreamPos stream_snap(int g, int t, int nt, int rows) {
  const int bt = unit_log2(rows, nt) + split_waves_log2(rows), s = ((t + (1 << bt) - 1) >> bt) << bt;
  return s >= nt ? StreamPos{g + 1, 0} : StreamPos{g, s};
}

// Blocks [beg, end) of share w of the line of the launch's tiles (every group's tiles, group after group): those that
// start in the w-th of 1 << logw equal parts of it.
__device__ __forceinline__ void stream_share(const KeySplitArgs& a, int rows, uint32_t w, StreamPos& beg,
                                             StreamPos& end) {
  const int lane = threadIdx.x & 63;
  if (!a.lens) {
    const int nt = tiles_of(a.L);
    const uint64_t total = (uint64_t)a.ngrp * (uint32_t)nt;
    auto find = [&](uint32_t i) {
      const uint64_t x = (total * i) >> a.logw;
      if (x >= total) return StreamPos{a.g0 + a.ngrp, 0};
      const uint64_t g = (x >> 32) ? x / (uint32_t)nt : (uint64_t)((uint32_t)x / (uint32_t)nt);
      return stream_snap(a.g0 + (int)g, (int)(x - g * (uint32_t)nt), nt, rows);
    };
    beg = find(w);
    end = find(w + 1);
    return;
  }
  // Ragged lengths: lane i of chunk c holds request 64 c + i; a group line of B * Hkv groups, b-major.
  auto chunk = [&](int c, uint32_t& nt) {
    const int b = 64 * c + lane;
    nt = b < a.B ? (uint32_t)tiles_of(stream_len(a, b)) : 0u;
    return wave_incl_scan(nt);
  };
  const int nc = (a.B + 63) / 64;
  uint32_t nt0;
  const uint32_t incl0 = chunk(0, nt0);
  uint64_t heads = __builtin_amdgcn_readlane(incl0, 63);    // tiles of one KV head over all requests
  for (int c = 1; c < nc; ++c) {
    uint32_t nt;
    heads += __builtin_amdgcn_readlane(chunk(c, nt), 63);
  }
  const uint64_t total = heads * (uint32_t)a.Hkv;
  auto find = [&](uint32_t i) {
    const uint64_t x = (total * i) >> a.logw;
    uint64_t run = 0;
    for (int c = 0; c < nc; ++c) {
      uint32_t nt = nt0, incl = incl0;
      if (c) incl = chunk(c, nt);
      const uint64_t m = __builtin_amdgcn_ballot_w64((run + incl) * (uint32_t)a.Hkv > x);
      if (m) {
        const int l = (int)__builtin_ctzll(m);
        const uint32_t ntb = __builtin_amdgcn_readlane(nt, l);
        const uint64_t rel = x - (run + __builtin_amdgcn_readlane(incl, l) - ntb) * (uint32_t)a.Hkv;
        const uint32_t h = (rel >> 32) ? (uint32_t)(rel / ntb) : (uint32_t)rel / ntb;
        return stream_snap((64 * c + l) * a.Hkv + (int)h, (int)(rel - (uint64_t)h * ntb), (int)ntb, rows);
      }
      run += __builtin_amdgcn_readlane(incl, 63);
    }
    return StreamPos{a.B * a.Hkv, 0};
  };
  beg = find(w);
  end = find(w + 1);
}

// ---- key sources: where the DMA finds tile t of group g.  Contiguous caches, or a page pool (PagedSrc's window of 64
// tiles, rebuilt when the walk leaves it).
constexpr int kStreamContig = 0, kStreamHND = 1, kStreamNHD = 2;

struct ContigTiles {
  const f16* kb;
  const f16* vb;
  int kend;
  static constexpr bool kStrided = false;   // rows 256 bytes apart
  __device__ const f16* ktile(int key0) const { return kb + (size_t)key0 * 128; }
  __device__ const f16* vtile(int key0) const { return vb + (size_t)key0 * 128; }
};

// The DMA cursor: the next tile to request, ahead of the tile being computed.  A wave's tiles in a group are those of
// its unit index u modulo q.
template <int kSrc>
struct StreamDma {
  int g, t, nt, n;
  StreamPos end;
  ContigTiles ct;
  PagedSrc<kSrc == kStreamNHD> pg;
  int wend;                // paged: first tile past the window

  __device__ __forceinline__ bool done() const { return g > end.g || (g == end.g && t >= end.t); }
  __device__ __forceinline__ void enter(const KeySplitArgs& a) {
    const int b = g / a.Hkv;
    n = stream_len_uniform(a, b);
    nt = tiles_of(n);
    if constexpr (kSrc == kStreamContig) {
      const size_t off = (size_t)g * a.L * 128;
      ct.kb = a.k + off;
      ct.vb = a.v + off;
      ct.kend = n;
    } else {
      wend = 0;                                             // no window of this group yet
    }
  }
  // To the next group with a tile of unit index u, or the end.
  __device__ __forceinline__ void settle(const KeySplitArgs& a, int u) {
    while (t >= nt) {
      ++g;
      t = u;
      if (done()) return;
      enter(a);
    }
  }
  // Requests the tile and steps past it; returns whether the tile's page is present.
  __device__ __forceinline__ bool issue(const KeySplitArgs& a, char* __restrict__ stage, const TileLanes& tl, int lane,
                                        int u, int q) {
    bool here = true;
    if constexpr (kSrc == kStreamContig) {
      issue_tile_dma(stage, ct, t * kTile, tl, lane);
    } else {
      if (t >= wend) {
        const int b = g / a.Hkv;
        pg = paged_src<kSrc == kStreamNHD>(a.k, a.v, a.ps, a.Hkv, a.num_pages, a.sl2,
                                           a.pages + (size_t)b * a.max_pages, a.max_pages, g - b * a.Hkv, t * kTile,
                                           min(n, (t + 64) * kTile));
        wend = t + 64;
      }
      here = pg.present(t * kTile);
      issue_tile_dma(stage, pg, t * kTile, tl, lane);
    }
    t += q;
    settle(a, u);
    return here;
  }
};

// The draft mask of this lane's row on the last kd positions, as up to kMaskWords 32-bit words (kd <= 32 * kMaskWords).
constexpr int kMaskWords = 8;
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));

// The mask words are a vector value, not an array: an array member makes the compiler keep the whole struct in LDS
// and fetch the words one dependent round trip at a time before the first tile.
struct DraftMask {
  u32x8 mw;          // the row's mask words; words at or past nw are not used
  int nw;
  __device__ uint32_t bit(int j) const {          // bit j of the row's mask, 0 <= j < 32 * kMaskWords
    const int wi = j >> 5;
    uint32_t w = mw[0];
#pragma unroll
    for (int i = 1; i < kMaskWords; ++i) w = wi == i ? mw[i] : w;
    return wi < nw ? (w >> (j & 31)) & 1u : 0u;
  }
  // Loads the nw (1 .. kMaskWords) mask words at mrow; every address stays inside the row.  mrow == null: the whole
  // tail is visible.
  __device__ void load(const uint32_t* mrow, int n) {
    if (!mrow) {
      nw = kMaskWords;
#pragma unroll
      for (int i = 0; i < kMaskWords; ++i) mw[i] = ~0u;
      return;
    }
    nw = n;
#pragma unroll
    for (int i = 0; i < kMaskWords; ++i) mw[i] = ldg4(mrow + min(i, n - 1));
  }
};

// What compute_tile_lds needs of the tile's group: length, mask, scale.
template <bool kBits>
struct StreamMask {
  DraftMask dm;
  int kend, tail0;
  bool here;               // the tile's page is present
  float scale;
  __device__ void mask(floatx16& s, int key0, int g) const {
    if (here && key0 + kTile <= (kBits ? tail0 : kend)) return;    // whole tile visible (same for the whole wave)
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int key = key0 + 8 * blk + 4 * g + c;
        bool ok = here && key < kend;
        if constexpr (kBits) ok = ok && ((key < tail0) | dm.bit(max(key - tail0, 0))) != 0u;
        s[4 * blk + c] = ok ? s[4 * blk + c] : kNegInf;
      }
  }
};

// Consumes loaded operands here, so that the compiler's wait for them stands at this point and not in front of every
// use in the tile loop, where it would drain the ring.
template <class V>
__device__ __forceinline__ void land(V (&qb)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(qb[i]));
}

// One wave's part of a share: unit u of q in each of the blocks [beg, end), through its private ring of NS stages
// (NS - 1 tiles in flight while one is computed).  At a unit's end the partial is stored and the state starts anew;
// the ring runs on, its next tiles (of whatever unit or group) already requested.  The 16 O stores of a partial are
// vector-memory operations issued after the tiles in flight, so the next wait allows for them instead of waiting for
// their completion.
template <int NS, int kSrc, bool kBits, class V>
__device__ __forceinline__ void stream_walk(const KeySplitArgs& a, char* __restrict__ ring,
                                            const char* __restrict__ base, uint32_t ring_off, StreamPos beg,
                                            StreamPos end, int u, int q, int rb) {
  const int lane = threadIdx.x & 63, r = lane & 31, gl = lane >> 5;
  const int R = a.kd * a.G, row = rb * 32 + r;
  const bool valid = row < R;
  const int di = (valid ? row : 0) / a.G, gg = (valid ? row : 0) - di * a.G;
  const int nvalid = R - rb * 32;
  StreamDma<kSrc> dma;
  dma.g = beg.g;
  dma.t = beg.t + u;
  dma.end = end;
  if (dma.done()) return;
  dma.enter(a);
  dma.settle(a, u);
  if (dma.done()) return;
  V qb[8];
  StreamMask<kBits> cm;
  cm.scale = a.sl2;
  int cg = dma.g, ct = dma.t, cnt, unit, uend, bt;         // bt: tiles of a block, log2
  auto unit_at = [&]() {                                    // the unit of tile ct, and the first tile past its block
    const int blk = ct >> bt;
    unit = blk * q + u;
    uend = min(cnt, (blk + 1) << bt);
  };
  auto enter = [&]() {                                      // the compute cursor enters group cg at tile ct
    const int b = cg / a.Hkv, h = cg - b * a.Hkv;
    load_qt(qb, a.q + ((size_t)(b * a.kd + di) * a.Hq + h * a.G + gg) * 128, gl, valid);
    if constexpr (kBits) cm.dm.load(a.bits ? a.bits + (size_t)(b * a.kd + di) * a.W : nullptr, a.W);
    cm.kend = stream_len_uniform(a, b);
    cm.tail0 = cm.kend - a.kd;
    cnt = tiles_of(cm.kend);
    bt = unit_log2(R, cnt) + split_waves_log2(R);
  };
  enter();
  unit_at();
  const TileLanes tl = tile_lanes(lane, ring_off);
  bool here[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) here[i] = true;
  int ahead = 0;                                            // tiles requested and not yet computed
  auto request = [&](auto S) {
    if (dma.done()) return false;
    here[S] = dma.issue(a, ring + S * kStageBytes, tl, lane, u, q);
    ++ahead;
    return true;
  };
  unroll_while<0, NS - 1>(request);
  land(qb);
  RowState st;
  row_state_init(st);
  bool stored = false;                                      // a partial was stored since the last wait
  while (true) {
    auto step = [&](auto S) {
      if (ahead == 0) return false;
      asm volatile("" ::: "memory");
      // Stage (S + NS - 1) % NS last held the previous tile, whose LDS reads all returned before its MFMAs used them.
      request(std::integral_constant<int, (S + NS - 1) % NS>());
      wait_vmem_dyn(16 * (ahead - 1) + (NS == 2 && stored ? 16 : 0));
      stored = false;
      cm.here = here[S];
      compute_tile_lds(st, qb, base + S * kStageBytes, tl, cm, ct * kTile, lane);
      ct += q;
      --ahead;
      if (ct >= uend) {
        const size_t slot = ((size_t)(cg - a.g0) * a.nrb + rb) * a.slots + unit;
        store_sums(reinterpret_cast<float*>(a.part_o) + slot * a.rows_s * 128, a.part_ml + slot * a.rows_s * 2, st, lane,
                   nvalid);
        stored = true;
        row_state_init(st);
        if (ahead > 0) {
          if (ct >= cnt) {                                  // the next group with a tile of this unit index
            do {
              ++cg;
              cnt = tiles_of(stream_len_uniform(a, cg / a.Hkv));
            } while (u >= cnt);
            ct = u;
            enter();
            land(qb);
            stored = false;                                 // the wait for q was a wait for the stores, too
          }
          unit_at();
        }
      }
      return true;
    };
    if (!unroll_while<0, NS>(step)) break;
  }
}

// NS stages per wave, 8 / NS waves per workgroup (128 KB of ring: one workgroup per CU).  Four waves of two stages
// hide each other's LDS and MFMA latency when the launch has waves enough; two waves of four stages serve the calls
// that do not.
template <int NS, int kSrc, bool kBits, class V>
__global__ __launch_bounds__(64 * 8 / NS) void key_units_kernel(KeySplitArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[8 * kStageBytes];
  constexpr int NW = 8 / NS;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t gw = blockIdx.x * NW + wave, w = gw >> 2;  // four waves to a share
  if (w >> a.logw) return;
  const int R = a.kd * a.G, q = split_waves(R), k = gw & 3;
  const int rb = q == 4 ? 0 : k & 1, u = q == 4 ? k : k >> 1;   // row blocks of one unit are neighbours
  StreamPos beg, end;
  stream_share(a, R, w, beg, end);
  beg.g = __builtin_amdgcn_readfirstlane(beg.g);
  beg.t = __builtin_amdgcn_readfirstlane(beg.t);
  end.g = __builtin_amdgcn_readfirstlane(end.g);
  end.t = __builtin_amdgcn_readfirstlane(end.t);
  const uint32_t ring_off = (uint32_t)wave * NS * kStageBytes;
  stream_walk<NS, kSrc, kBits, V>(a, smem + ring_off, smem, ring_off, beg, end, u, q, rb);
}

// ---- one workgroup per split, the units folded in registers.
template <bool kBits>
struct SplitSrc {
  ContigTiles ct;
  StreamMask<kBits> cm;
  int kend;
  float scale;
  static constexpr bool kStrided = false;
  __device__ const f16* ktile(int key0) const { return ct.ktile(key0); }
  __device__ const f16* vtile(int key0) const { return ct.vtile(key0); }
  __device__ void mask(floatx16& s, int key0, int g) const { cm.mask(s, key0, g); }
};

// kFinal: no group has more than one split; its rows are the result and no combine launch follows.  (The combines of
// larger caches write a group's only split as it is, too: the same bits.)  Decode of one and 16 requests of 1000 keys
// 15.3 and 16.6 us with the combine, 12.2 and 13.7 without; verification of 16 drafts in four of 2000 keys 35.3 and
// 32.4.
//
// Ragged lengths: workgroup id i runs on XCD i modulo 8, so with eight splits to a group (16384 positions) split 7 of
// every group, which only the longest requests have, would run on one XCD and split 0, which all have, on another.  The
// splits of each next group that starts on the same XCD are therefore rotated by one.  Lengths of 1/16 to all of the
// cache, us, without and with: 4 rows, 8 requests in 16384 positions 63.6 and 46.9; 24 rows (4 KV heads), 64 requests
// 266 and 213; 32 rows (2 KV heads), 32 requests 69.3 and 57.6.  Split-major order balances as well, but leaves the
// workgroups without keys for the end: 8 requests in 32768 positions 126 against 119.
template <int kSrc, bool kBits, class V, bool kFinal>
__global__ __launch_bounds__(256) void key_split_kernel(KeySplitArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[kAttnSmemBytes];
  const int grel = blockIdx.x / a.slots;
  int split = blockIdx.x - grel * a.slots;
  if (a.lens) {
    split += (grel >> (3 - min(3, __builtin_ctz(a.slots)))) % a.slots;
    if (split >= a.slots) split -= a.slots;
  }
  const int item = grel * a.slots + split;                  // where the partial goes
  const int g = a.g0 + grel, b = g / a.Hkv, h = g - b * a.Hkv;
  const int R = a.kd * a.G, n = stream_len_uniform(a, b), keys = split_log2(R, n), kbeg = split << keys;
  const int kend = min(n, kbeg + (1 << keys)), ntiles = kbeg < n ? tiles_of(kend - kbeg) : 0;
  const int unit = unit_tiles(R, tiles_of(n));
  auto qrow = [&](int r) {
    const int i = r / a.G, gg = r - i * a.G;
    return a.q + ((size_t)(b * a.kd + i) * a.Hq + h * a.G + gg) * 128;
  };
  typedef part_t<elem_t<V>> PT;
  constexpr bool kDual = kSrc == kStreamContig && sizeof(PT) == 2;   // pages have at most 16 rows
  char* const po_b = reinterpret_cast<char*>(a.part_o) + (size_t)item * a.rows_s * 128 * a.esize;
  std::conditional_t<kDual, HalfOrFloat, PT*> po;
  if constexpr (kDual)
    po = HalfOrFloat{po_b, split_wide(R, n)};
  else
    po = reinterpret_cast<PT*>(po_b);
  float* pml = a.part_ml + (size_t)item * a.rows_s * 2;
  auto orow = [&](int r) {
    const int i = r / a.G, gg = r - i * a.G;
    return reinterpret_cast<elem_t<V>*>(a.out) + ((size_t)(b * a.kd + i) * a.Hq + h * a.G + gg) * 128;
  };
  auto attend = [&](const auto& src) {
    const auto run = [&](auto WR) {
      constexpr int kWR = decltype(WR)::value;
      if constexpr (kFinal)
        attend_wg<kWR, 4 / kWR, 2, V, true>(smem, src, qrow, R, kbeg, ntiles, po, pml, unit, orow);
      else
        attend_wg<kWR, 4 / kWR, 2, V, true>(smem, src, qrow, R, kbeg, ntiles, po, pml, unit);
    };
    if (kBits && R > 32)                                    // decode with more than 32 rows takes kBits, too
      run(std::integral_constant<int, 2>());
    else
      run(std::integral_constant<int, 1>());
  };
  if constexpr (kSrc == kStreamContig) {
    SplitSrc<kBits> src;
    const size_t off = (size_t)g * a.L * 128;
    src.ct.kb = a.k + off;
    src.ct.vb = a.v + off;
    src.kend = kend;
    src.scale = a.sl2;
    src.cm.kend = kend;
    src.cm.tail0 = n - a.kd;
    src.cm.here = true;
    if constexpr (kBits) {
      const int lrow = (threadIdx.x & 31) + (R > 32 ? 32 * ((threadIdx.x >> 6) & 1) : 0);
      const int di = (lrow < R ? lrow : 0) / a.G;
      src.cm.dm.load(a.bits ? a.bits + (size_t)(b * a.kd + di) * a.W : nullptr, a.W);
    }
    attend(src);
  } else {
    attend(paged_src<kSrc == kStreamNHD>(a.k, a.v, a.ps, a.Hkv, a.num_pages, a.sl2,
                                         a.pages + (size_t)b * a.max_pages, a.max_pages, h, kbeg, kend));
  }
}

// The final merge of a row's splits: combine_row's arithmetic (split 0 first) over the splits in use.  An only split is
// the result, rounded once as key_split_kernel writes it where the cache holds no second one (a bf16 row weighed and
// divided again could round to the other side).
template <class E>
__global__ __launch_bounds__(128) void key_split_combine_kernel(KeySplitArgs a) {
  const int R = a.kd * a.G;
  const int grel = blockIdx.x / R, row = blockIdx.x - grel * R;
  const int g = a.g0 + grel, b = g / a.Hkv, h = g - b * a.Hkv;
  const int len = stream_len_uniform(a, b), n = group_splits(R, len);
  const int i = row / a.G, gg = row - i * a.G;
  E* out = reinterpret_cast<E*>(a.out) + ((size_t)(b * a.kd + i) * a.Hq + h * a.G + gg) * 128;
  auto merge = [&](auto t) {
    typedef decltype(t) T;
    auto part = [&](int s, const float*& ml, const T*& o) {
      const size_t item = (size_t)grel * a.slots + s;
      ml = a.part_ml + (item * a.rows_s + row) * 2;
      o = reinterpret_cast<const T*>(reinterpret_cast<const char*>(a.part_o) + item * a.rows_s * 128 * a.esize) +
          row * 128;
    };
    if (n == 1) {
      const float* ml;
      const T* o;
      part(0, ml, o);
      out[threadIdx.x] = (E)(ml[1] == 0.f ? __builtin_nanf("") : (float)o[threadIdx.x]);
    } else {
      combine_row<128, 1, T>(n, part, out);
    }
  };
  if (sizeof(part_t<E>) == 2 && split_wide(R, len))
    merge(float());
  else
    merge(part_t<E>());
}

// The same for many rows (at least kSplitVecRows): one wave per 4 rows, 16 lanes per row, each lane 8 head-dims loaded
// 16 bytes at a time, so the partials stream with a quarter of the load instructions per byte.  Same bits.
constexpr int kSplitVecRows = 1024;
template <class E>
__global__ __launch_bounds__(64) void key_split_combine_vec_kernel(KeySplitArgs a) {
  const int R = a.kd * a.G;
  const int lane = threadIdx.x, c = lane & 15;
  const int rowg = blockIdx.x * 4 + (lane >> 4);
  if (rowg >= a.ngrp * R) return;                           // a whole row group of lanes
  const int grel = rowg / R, row = rowg - grel * R;
  const int g = a.g0 + grel, b = g / a.Hkv, h = g - b * a.Hkv;
  const int len = stream_len(a, b), n = group_splits(R, len);
  const int i = row / a.G, gg = row - i * a.G;
  E* out = reinterpret_cast<E*>(a.out) + ((size_t)(b * a.kd + i) * a.Hq + h * a.G + gg) * 128 + 8 * c;
  auto merge = [&](auto t) {
    typedef decltype(t) T;
    auto part = [&](int s, const float*& ml, const T*& o) {
      const size_t item = (size_t)grel * a.slots + s;
      ml = a.part_ml + (item * a.rows_s + row) * 2;
      o = reinterpret_cast<const T*>(reinterpret_cast<const char*>(a.part_o) + item * a.rows_s * 128 * a.esize) +
          row * 128 + 8 * c;
    };
    if (n == 1) {
      const float* ml;
      const T* op;
      part(0, ml, op);
      Part8<T> o;
      o.load(op);
      const bool none = ml[1] == 0.f;
      float x[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = none ? __builtin_nanf("") : o.get(k);
      store_out8(out, x, 1.f);
    } else {
      combine_vec<T>(n, part, out);
    }
  };
  if (sizeof(part_t<E>) == 2 && split_wide(R, len))
    merge(float());
  else
    merge(part_t<E>());
}

// One output row per workgroup from stored units: lane group s (16 lanes, eight head-dims each) folds the units of
// split s + 16 j of each wave, merges the waves and rounds the split as key_split_kernel stores it; then 128 threads
// sum the splits, split 0 first, as combine_row does.
template <class E>
__global__ __launch_bounds__(256) void key_units_combine_kernel(KeySplitArgs a) {
  typedef part_t<E> PT;
  __shared__ float redm[4], sm[16], sl[16];
  __shared__ __attribute__((aligned(16))) float so_f[16 * 128];   // the splits' rows: fp32 if wide, else PT
  PT* const so_h = reinterpret_cast<PT*>(so_f);
  const int tid = threadIdx.x, c = tid & 15, s = tid >> 4;
  const int R = a.kd * a.G;
  const int grel = blockIdx.x / R, row = blockIdx.x - grel * R;
  const int g = a.g0 + grel, b = g / a.Hkv, h = g - b * a.Hkv;
  const int len = stream_len_uniform(a, b), nt = tiles_of(len), n = group_units(R, nt);
  // Waves of a split, and units of a wave in it.
  const int q = split_waves(R), per = 1 << (split_log2(R, len) - 5 - split_waves_log2(R) - unit_log2(R, nt));
  const int nsplit = group_splits(R, len);
  const bool wide = sizeof(PT) == 4 || split_wide(R, len);
  const size_t p0 = (((size_t)grel * a.nrb + (row >> 5)) * a.slots) * a.rows_s + (row & 31);
  const float* po = reinterpret_cast<const float*>(a.part_o) + 8 * c;
  auto ml_of = [&](int i) { return *reinterpret_cast<const float2*>(a.part_ml + (p0 + (size_t)i * a.rows_s) * 2); };
  // Split s0 + s: its waves' units folded and merged.
  auto split_state = [&](int sp) {
    float om[4][8], wm[4], wl[4];
    float M = kNegInf;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      wm[u] = kNegInf;
      wl[u] = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) om[u][k] = 0.f;
    }
    // Units of the split in order: unit e of wave u is sp * per * q + e * q + u.  All of one e in flight together, the
    // next e's requested before they are used.
    Part8<float> ov[4], nx[4];
    float2 mv[4], mx[4];
    auto fetch = [&](int e, Part8<float> (&o)[4], float2 (&m)[4]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = min((sp * per + min(e, per - 1)) * q + min(u, q - 1), n - 1);   // in bounds; unused past n
        m[u] = ml_of(i);
        o[u].load(po + (p0 + (size_t)i * a.rows_s) * 128);
      }
    };
    fetch(0, ov, mv);
    for (int e = 0; e < per; ++e) {
      if ((sp * per + e) * q >= n) break;
      fetch(e + 1, nx, mx);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u < q && (sp * per + e) * q + u < n) {
          if (e == 0) {
            wm[u] = mv[u].x;
            wl[u] = mv[u].y;
#pragma unroll
            for (int k = 0; k < 8; ++k) om[u][k] = ov[u].get(k);
          } else {
            const float Mf = fmaxf(wm[u], mv[u].x), ah = merge_scale(wm[u], Mf), au = merge_scale(mv[u].x, Mf);
#pragma unroll
            for (int k = 0; k < 8; ++k) om[u][k] = fold_val(ah, om[u][k], au, ov[u].get(k));
            wl[u] = fold_val(ah, wl[u], au, mv[u].y);
            wm[u] = Mf;
          }
        }
        ov[u] = nx[u];
        mv[u] = mx[u];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) M = fmaxf(M, wm[u]);
    float acc[8], l = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (u >= q) break;
      const float ak = merge_scale(wm[u], M);
      l = merge_add(l, ak, wl[u]);
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] = merge_add(acc[k], ak, om[u][k]);
    }
    const float inv = part_inv(l);
    if (c == 0) {
      sm[s] = M;
      sl[s] = l;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      acc[k] *= inv;
      asm("" : "+v"(acc[k]));                               // rounded to fp32 first, not fused with the conversion
    }
    auto put = [&](auto* so) {
#pragma unroll
      for (int k = 0; k < 8; k += 4)
        store_part4(so + s * 128 + 8 * c + k, floatx4{acc[k], acc[k + 1], acc[k + 2], acc[k + 3]});
    };
    if (wide)
      put(so_f);
    else
      put(so_h);
  };
  float M = kNegInf;
  if (nsplit > 16) {                                        // the largest m before the first weight
    for (int i = tid; i < n; i += 256) M = fmaxf(M, ml_of(i).x);
    M = wave_max(M);
    if ((tid & 63) == 0) redm[tid >> 6] = M;
  }
  float num = 0.f, den = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += 16) {
    if (s0) __syncthreads();
    if (s0 + s < nsplit) split_state(s0 + s);
    __syncthreads();
    const int ns = min(16, nsplit - s0);
    if (tid < 128) {
      if (s0 == 0) {
        if (nsplit > 16) {
          M = fmaxf(fmaxf(redm[0], redm[1]), fmaxf(redm[2], redm[3]));
        } else {
          for (int j = 0; j < ns; ++j) M = fmaxf(M, sm[j]);
        }
        M = (M == kNegInf) ? 0.f : M;
      }
      auto add = [&](const auto* so) {
        for (int j = 0; j < ns; ++j) {
          const float w = part_weight(float2{sm[j], sl[j]}, M);
          den += w;
          num += w * (float)so[j * 128 + tid];
        }
      };
      if (wide)
        add(so_f);
      else
        add(so_h);
    }
  }
  if (tid >= 128) return;
  if (nsplit == 1) {                                        // the split is the result, as key_split_kernel writes it
    num = sl[0] == 0.f ? __builtin_nanf("") : wide ? so_f[tid] : (float)so_h[tid];
    den = 1.f;
  }
  const int di = row / a.G, gg = row - di * a.G;
  reinterpret_cast<E*>(a.out)[((size_t)(b * a.kd + di) * a.Hq + h * a.G + gg) * 128 + tid] = (E)(num / den);
}

// ---- host side
struct KeySplitPlan {
  int rows, nsplit;        // nsplit: splits of a group of L keys
  bool units;
  int nrb, slots, rows_s;
  size_t esize;            // bytes for an element of a partial row
  size_t grp_rows;         // partial rows of one group
};

// Bytes of the O rows (to the next 256-byte boundary) and of all partials of ngrp groups.
inline size_t key_split_ml_offset(const KeySplitPlan& p, int64_t ngrp) {
  return (ngrp * p.grp_rows * 128 * p.esize + 255) / 256 * 256;
}
inline size_t key_split_bytes(const KeySplitPlan& p, int64_t ngrp) {
  return key_split_ml_offset(p, ngrp) + ngrp * p.grp_rows * 2 * sizeof(float);
}

// The most splits and rows of a unit launch.
inline int64_t unit_max_splits(int rows) { return kDeviceCUs / (rows > 32 ? 2 : 4); }
inline int64_t unit_max_rows(int rows) { return rows > 32 ? 1024 : 512; }

// Units while the splits of all groups (at their longest) leave three quarters of the CUs without one (half, with more
// than 32 rows, whose tiles cost two waves), there are units to deal out, and the rows are few enough that the units'
// stores and their merge do not cost more than the wider walk saves.  Measured, us, units against splits:
//   decode (8 KV heads of 4 rows), 1, 2, 4 requests of 8192 keys: 14.4, 18.4, 32.7 against 19.7, 19.7, 31.6; 8 of 2000
//   keys: 18.5 against 20.2; verification of 8 drafts, 1, 2, 4 requests of 8192 keys: 16.9, 21.3, 40.1 against 30.8,
//   30.8, 33.4, and 8 of 1000 keys: 20.9 against 16.1; of 16 drafts (64 rows), 1, 2 requests of 32768 keys: 38, 72
//   against 82, 82, and 8 of 1000 keys: 31.2 against 21.5.
// A cache of one split of at most ten tiles to a wave is never dealt out: the split alone is one launch.  Decode of one
// and eight requests of 1000 keys 15.3 and 14.7 us as units, 12.2 and 12.1 as a split; of one of 1500 keys 15.0 and
// 15.3, of 2048 15.0 and 18.6.
//
// ragged: a group may be shorter than L (and have more splits than one of L keys, where the split size steps up). e:
// bytes of an element of a split's row (fp32 for fp16 inputs where split_wide() can hold).  room: bytes there are for
// the partials of all groups; units that need more stay splits, with the same bits.
inline KeySplitPlan key_split_plan(int64_t ngrp, int64_t rows, int64_t L, bool ragged, size_t e, size_t room) {
  KeySplitPlan p;
  p.rows = (int)rows;
  p.nsplit = (int)group_splits((int)rows, L);
  const int64_t nt = (L + kTile - 1) / kTile;
  p.units = ngrp * p.nsplit <= unit_max_splits(p.rows) && ngrp * rows <= unit_max_rows(p.rows) &&
            nt > split_waves(p.rows) * unit_tiles(p.rows, (int)nt) &&
            (p.nsplit > 1 || nt > 10 * split_waves(p.rows));
  auto lay_out = [&] {
    p.nrb = p.units ? (int)((rows + 31) / 32) : 1;
    p.rows_s = rows <= 32 || !p.units ? (int)rows : 32;
    p.slots = (int)(p.units ? unit_slots((int)rows, L) : ragged ? split_slots((int)rows, L) : p.nsplit);
    p.esize = p.units || (rows > 16 && (ragged ? L > 2048 : split_wide((int)rows, L))) ? sizeof(float) : e;
    p.grp_rows = (size_t)p.nrb * p.slots * p.rows_s;
  };
  lay_out();
  if (p.units && key_split_bytes(p, ngrp) > room) {
    p.units = false;
    lay_out();
  }
  return p;
}

// Bytes of partials, in fp32, that hold those of any call of up to ngrp groups over caches of up to L positions, so
// that one workspace sized for the largest call serves the smaller ones: a call of fewer groups may take units, which
// need more than the splits of many groups do.  A unit launch has at most unit_max_splits() splits and unit_max_rows()
// rows, and a group at most 64 units or split_waves() to a split.
inline size_t key_split_max_bytes(int64_t ngrp, int64_t rows64, int64_t L) {
  const int rows = (int)rows64, q = split_waves(rows);
  const int64_t cap = std::min(ngrp, std::min(unit_max_splits(rows), unit_max_rows(rows) / rows));
  const int64_t units = std::max(cap * std::min<int64_t>(64, (L + kTile - 1) / kTile),
                                 q * std::min(unit_max_splits(rows), ngrp * split_slots(rows, L)));
  const size_t unit_rows = (size_t)units * ((rows + 31) / 32) * (rows <= 32 ? rows : 32);
  const size_t split_rows = (size_t)ngrp * split_slots(rows, L) * rows;
  return std::max(unit_rows, split_rows) * (128 + 2) * sizeof(float) + 256;
}

// Partial and combine launches over the groups [a.g0, a.g0 + a.ngrp), partials at `partials`
// (key_split_bytes(p, a.ngrp, ..) bytes, 256-byte aligned, uninitialised).
template <int kSrc, bool kBits, class V>
inline int key_split_launch(KeySplitArgs a, const KeySplitPlan& p, void* partials, hipStream_t s) {
  typedef elem_t<V> E;
  a.part_o = partials;
  a.part_ml = reinterpret_cast<float*>((char*)partials + key_split_ml_offset(p, a.ngrp));
  a.nrb = p.nrb; a.slots = p.slots; a.rows_s = p.rows_s; a.esize = (int)p.esize;
  const int64_t rows = (int64_t)a.ngrp * p.rows;
  if (!p.units) {
    prof_before(kKSpecPartial, s);
    if (p.nsplit == 1)
      hipLaunchKernelGGL((key_split_kernel<kSrc, kBits, V, true>), dim3((unsigned)a.ngrp), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((key_split_kernel<kSrc, kBits, V, false>), dim3((unsigned)(a.ngrp * p.slots)), dim3(256), 0, s,
                         a);
    prof_after(kKSpecPartial, s);
    VMK_CHECK_HIP(hipGetLastError());
    if (p.nsplit == 1) {
      prof_before(kKSpecCombine, s);                        // an armed bracket closes over nothing
      prof_after(kKSpecCombine, s);
      return 0;
    }
    prof_before(kKSpecCombine, s);
    if (rows >= kSplitVecRows)
      hipLaunchKernelGGL(key_split_combine_vec_kernel<E>, dim3((unsigned)((rows + 3) / 4)), dim3(64), 0, s, a);
    else
      hipLaunchKernelGGL(key_split_combine_kernel<E>, dim3((unsigned)rows), dim3(128), 0, s, a);
  } else {
    const int64_t nt = (a.L + (int64_t)kTile - 1) / kTile;
    const int64_t bt = split_waves(p.rows) * unit_tiles(p.rows, (int)nt);
    const int64_t blocks = (int64_t)a.ngrp * ((nt + bt - 1) / bt);
    // Shares of four waves: a power of two, at least one per block up to four waves on every CU.  Two waves of four
    // stages per workgroup while that leaves CUs free.
    const bool deep = 2 * blocks <= kDeviceCUs;
    const int nw = deep ? 2 : 4;
    a.logw = 0;
    while ((1 << a.logw) < blocks && (4 << a.logw) < nw * kDeviceCUs) ++a.logw;
    const unsigned grid = (unsigned)((4 << a.logw) / nw);
    prof_before(kKSpecPartial, s);
    if (deep)
      hipLaunchKernelGGL((key_units_kernel<4, kSrc, kBits, V>), dim3(grid), dim3(128), 0, s, a);
    else
      hipLaunchKernelGGL((key_units_kernel<2, kSrc, kBits, V>), dim3(grid), dim3(256), 0, s, a);
    prof_after(kKSpecPartial, s);
    VMK_CHECK_HIP(hipGetLastError());
    prof_before(kKSpecCombine, s);
    hipLaunchKernelGGL(key_units_combine_kernel<E>, dim3((unsigned)rows), dim3(256), 0, s, a);
  }
  prof_after(kKSpecCombine, s);
  VMK_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace vmk
