// scatter_add over one axis: out[p, k, q] = in[p, k, q] + the updates u[p, j, q] of every j whose clamped
// index is k, added in the order of j (src/tensor/lower.zig's order, which rounds every sum), in one pass
// over the table: each row of it is read once and written once, and the updates of a row are added in
// registers.
//
// What bounds it is the table's copy (read and write of every row) and the updates read once; the
// rows that many updates hit (a frequent token) are the serial part, so their updates are loaded
// eight to 32 at a time (32 registers' worth) ahead of the dependent additions. One thread per (p, q) walking all j, as before,
// took 1004 us a pass for 4096 updates of a 32000 x 1024 f32 table, the 43 us copy of the table among them (1390 as
// PyTorch's wheel compiles it): one dependent load, add and store per update and only 1024 threads in flight.
//
// A workgroup owns ROWS = LOOP x 4 x KG rows of PG x PLOOP positions of p and one tile of q: LOOP x 4 blocks of KG
// consecutive rows, ROW_TILES blocks apart, so that the frequent tokens, whose ids are small in most
// vocabularies, fall to different workgroups (four consecutive rows per workgroup took 194 us
// instead of 87 us for the table above, now 66-78, with ids whose frequency falls as 1 / rank). It
// reads the whole index list (from L2) and keeps the entries of its rows: (row, j) pairs in LDS, in
// the order of j (ballot ranks). A batch of up to CAP of them is sorted stably by row (the rank of every key among
// the batch: keys are row * CAP + position, all distinct), and each group of TC threads (along a row) then adds
// the runs of its four rows. The lists are the same for every p: where KG groups cover the rows of one, the workgroup's
// other groups take the next PG - 1 positions, and all of them PLOOP positions in turn. (1048576 x 8 f32 with
// 64 updates along the last axis: 5886 us with a workgroup for every p, now 150; 300 with a thread for every p.)
// When more entries remain, the next batch continues from the rows just written (the same thread wrote them).
//
// S supplies the sizes (NI updates, EXT rows, POST elements per row, PRE), TC, KG, LOOP, PLOOP, VEC (4 when POST
// is a multiple of it), index(j), plus(a, u), and on the VEC elements c0 .. c0 + VEC - 1 of a row
// init(p, k, c0, v), again(p, k, c0, v), update(p, j, c0, v) and store(p, k, c0, v).
#pragma once

namespace accy {
namespace scatter {

struct alignas(16) Int4 { int v[4]; };

constexpr int BLOCK = 256, RR = 4, CAP = 1024, STEP = 512;  // STEP indices per scan round (two per thread)

// Adds the updates of sorted[x .. e - 1], at most N, in order: N loads (past the end the last one again,
// not added), then the additions.
template <int N, class S, class I, class T>
__device__ __forceinline__ void add_run(const S& s, const I* sorted, int x, int e, I p, I c0, T (&v)[S::VEC]) {
  T u[N][S::VEC];
#pragma unroll
  for (int i = 0; i < N; ++i) s.update(p, sorted[x + i < e ? x + i : e - 1], c0, u[i]);
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int w = 0; w < S::VEC; ++w) v[w] = x + i < e ? S::plus(v[w], u[i][w]) : v[w];
}

template <class S>
__device__ __forceinline__ void rows(const S& s) {
  typedef typename S::I I;
  typedef typename S::T T;
  constexpr int VEC = S::VEC, LOOP = S::LOOP;
  constexpr long VECS = S::POST / VEC;
  constexpr int TC = S::TC, KG = S::KG, PG = BLOCK / TC / KG, ROWS = LOOP * KG * RR;
  constexpr int DEPTH = TC <= 64 ? 16 : 32 / VEC;
  constexpr long COL_TILES = (VECS + TC - 1) / TC, ROW_TILES = (S::EXT + ROWS - 1) / ROWS;  // blocks of KG rows a tile apart
  constexpr long TILES = ROW_TILES * COL_TILES * ((S::PRE + PG * S::PLOOP - 1) / (PG * S::PLOOP));
  static_assert(PG * KG * TC == BLOCK, "whole groups");
  static_assert((long)ROWS * CAP < (1l << 31), "keys fit an int");
  __shared__ __attribute__((aligned(16))) int key[CAP];
  __shared__ int row_of[CAP];
  __shared__ I pos[CAP], sorted[CAP];
  __shared__ int first[ROWS], last[ROWS];
  __shared__ int wave_count[BLOCK / 64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int group = PG > 1 ? tid / TC % KG : tid / TC;
  for (long tile = blockIdx.x; tile < TILES; tile += gridDim.x) {
    const I mine = (I)(tile % ROW_TILES);
    // local row (block i, group g) <-> row of the table
    auto row_at = [&](int i, int g) { return ((I)i * (I)ROW_TILES + mine) * KG + g; };
    const I p0 = (I)(tile / ROW_TILES / COL_TILES) * (PG * S::PLOOP) + (PG > 1 ? tid / TC / KG : 0);
    const I c0 = ((I)(tile / ROW_TILES % COL_TILES) * TC + (I)(tid % TC)) * VEC;
    const bool in_row = c0 < (I)S::POST;
    // the last workgroup's positions may reach past the end
    auto exists = [](I p) { return PG * S::PLOOP == 1 || p < (I)S::PRE; };
    T v[RR][VEC];
    // The first rows of the tile are loaded before the scan, so that the scan hides their latency.
#pragma unroll
    for (int i = 0; i < RR; ++i) {
      const I k = row_at(i, group);
      if (in_row && exists(p0) && k < (I)S::EXT) s.init(p0, k, c0, v[i]);
    }
    I next = 0;
    bool begun = false;
    do {
      int n = 0;  // entries in this batch (the same in every thread)
      while (next < (I)S::NI && n <= CAP - STEP) {
        // wave w tests indices next + 128 w .. + 127, so ranks follow j
        int row[2];
        u64_t hits[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const I j = next + wave * 128 + h * 64 + lane;
          const I k = j < (I)S::NI ? s.index(j) : (I)0;
          const I block = k / KG;
          const bool hit = j < (I)S::NI && block % (I)ROW_TILES == mine;
          row[h] = hit ? (int)(block / (I)ROW_TILES) * KG + (int)(k % KG) : -1;
          hits[h] = __ballot(hit);
        }
        if (lane == 0) wave_count[wave] = __popcll(hits[0]) + __popcll(hits[1]);
        __syncthreads();
        int at = n;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; ++w) {
          if (w < wave) at += wave_count[w];
          n += wave_count[w];
        }
        const u64_t below = (1ull << lane) - 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (row[h] >= 0) {
            const int e = at + __popcll(hits[h] & below);
            key[e] = row[h] * CAP + e;
            pos[e] = next + wave * 128 + h * 64 + lane;
          }
          at += __popcll(hits[h]);
        }
        next += STEP;
        __syncthreads();
      }
      if (n) {
        for (int i = tid; i < ROWS; i += BLOCK) first[i] = last[i] = 0;
        if (tid < 4 && n + tid < CAP) key[n + tid] = 0x7fffffff;  // fills the last vector of four
        __syncthreads();
        // Every key's rank, CAP / BLOCK keys per thread against four at a time. (One at a time, each read waited
        // for: 190 us for 8000 updates of a 50000 x 256 table,
        // whose frequent rows one workgroup takes, now 76.)
        int own[CAP / BLOCK], rank[CAP / BLOCK];
#pragma unroll
        for (int h = 0; h < CAP / BLOCK; ++h) {
          own[h] = tid + h * BLOCK < n ? key[tid + h * BLOCK] : 0;
          rank[h] = 0;
        }
#pragma unroll 2
        for (int i = 0; i < n; i += 4) {
          const Int4 other = *(const Int4*)(key + i);
#pragma unroll
          for (int h = 0; h < CAP / BLOCK; ++h)
#pragma unroll
            for (int w = 0; w < 4; ++w) rank[h] += other.v[w] < own[h] ? 1 : 0;
        }
#pragma unroll
        for (int h = 0; h < CAP / BLOCK; ++h)
          if (tid + h * BLOCK < n) {
            sorted[rank[h]] = pos[tid + h * BLOCK];
            row_of[rank[h]] = own[h] / CAP;
          }
        __syncthreads();
        for (int x = tid; x < n; x += BLOCK) {
          const int r = row_of[x];
          if (x == 0 || row_of[x - 1] != r) first[r] = x;
          if (x + 1 == n || row_of[x + 1] != r) last[r] = x + 1;
        }
        __syncthreads();
      }
      auto add = [&](I p, bool loaded) {
        for (int t = 0; t < LOOP; ++t) {
#pragma unroll
          for (int i = 0; i < RR; ++i) {
            const I k = row_at(t * RR + i, group);
            if (!in_row || !exists(p) || k >= (I)S::EXT) continue;
            const int r = (t * RR + i) * KG + group;
            int x = n ? first[r] : 0;
            const int e = n ? last[r] : 0;
            if (begun) {
              if (x == e) continue;
              s.again(p, k, c0, v[i]);
            } else if (t > 0 || !loaded) {
              s.init(p, k, c0, v[i]);
            }
            for (; e - x > 4; x += DEPTH) add_run<DEPTH>(s, sorted, x, e, p, c0, v[i]);
            if (x < e) add_run<4>(s, sorted, x, e, p, c0, v[i]);
            s.store(p, k, c0, v[i]);
          }
        }
      };
      add(p0, true);
#pragma unroll 1
      for (int pl = 1; pl < S::PLOOP; ++pl) add(p0 + pl * PG, false);
      begun = true;
      __syncthreads();  // the lists are rewritten by the next batch
    } while (next < (I)S::NI);
  }
}

}  // namespace scatter
}  // namespace accy
