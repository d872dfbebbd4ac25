// chunks.h -- how the k-marching launches cut their planes into chunks (host code).
#pragma once

namespace tosca {

constexpr int NUM_CU = 256;

// What a marching kernel's chunks depend on: the workgroups a compute unit runs at a time, the plane steps
// a workgroup primes its registers and LDS with, and how soon neighbouring tiles stop sharing their halo
// lines (a launch costs 1 + planes / drift per step).
struct ChunkRule { int per_cu, over; double drift; };
constexpr ChunkRule CHUNK_FORMU{1, 3, 2000.0};
constexpr ChunkRule CHUNK_FILTER3{1, 3, 2e4};
constexpr ChunkRule CHUNK_FILTER5{1, 5, 2e4};
constexpr ChunkRule CHUNK_FILTER_F32{1, 2, 2e4};
constexpr ChunkRule CHUNK_BOX{2, 2, 500.0};
constexpr ChunkRule CHUNK_DPASD_IJ{1, 1, 2000.0};
constexpr ChunkRule CHUNK_DPASD_K{4, 2, 500.0};
constexpr ChunkRule CHUNK_VJP_MARCH{2, 3, 2000.0};
constexpr ChunkRule CHUNK_VJP_FINISH{2, 2, 500.0};
constexpr ChunkRule CHUNK_FORMT{2, 1, 500.0};

// k planes per chunk of a k-marching launch over `tiles` column tiles.  Workgroups run `slots` at a
// time, each for its planes plus `over` plane steps of priming, so the launch takes about
// ceil(tiles chunks / slots) (planes + over) plane steps, and neighbouring tiles drift apart along k,
// so that they share fewer of their halo lines in L2: 1 + planes / drift per step.  The chunk count
// that makes the product least, the smallest one where several do.  Large grids get whole rounds of
// the chip (the 512 x 512 x 192 shard: FormU 8 chunks of 64 planes, 7.9 rounds, 4.99 ms; 5.31 in one
// chunk, 5.42 in 24); grids with few columns get chunks short enough to occupy it (64^3 FormU 58 us,
// 69 with the 8-plane chunks it had; 256 x 128 x 96 hill 0.39 ms, 0.47; 16 x 10 x 8 hill 21 us, 65).
// Of the counts with the same planes per chunk only the first is looked at, about 2 sqrt(nk) in all: the
// caller waits for this on each launch (0.3 us for 192 planes, 1.5 for 4096; 1.3 and 26 over every count).
inline int plane_chunk(int nk, int tiles, ChunkRule r) {
    const long slots = (long)r.per_cu * NUM_CU;
    double best = -1.0;
    int kc = nk;
    for (int k = nk; k >= 1;) {
        const int n = (nk + k - 1) / k;
        k = (nk + n - 1) / n;
        const double cost = (double)(((long)tiles * n + slots - 1) / slots) * (k + r.over) * (1.0 + k / r.drift);
        if (best < 0.0 || cost < best) { best = cost; kc = k; }
        k--;
    }
    return kc;
}

}  // namespace tosca
