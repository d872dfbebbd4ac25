// chunks.h -- how the k-marching launches cut their planes into chunks (host code).
#pragma once

namespace tosca {

constexpr int NUM_CU = 256;

// What a marching kernel's chunks depend on: the workgroups a compute unit runs at a time, the plane steps
// a workgroup primes its registers and LDS with, and how soon neighbouring tiles stop sharing their halo
// lines (a launch costs 1 + planes / drift per step).
//
// per_cu is what the kernel's registers and LDS let a unit hold (CHUNK_DPASD_K: less than that), `over` its
// priming loop.  drift was set with the first measurements of each kernel and is worth a few per cent at
// most.  Kernel time with another constant over the time with the one here, geometric mean over nine grids
// (512 x 512 x 192, 384 x 256 x 128, 333 x 253 x 131, 256 x 192 x 96, 192 x 192 x 128, 128 x 96 x 64, 64^3,
// 512 x 62 x 18, 96 x 126 x 18), runs differing by 1 %:
//                  per_cu / 2   per_cu * 2   drift 100    500   2000    2e4   none
//     FORMU             -          1.09        1.02      1.00   1      1.00   1.00   (none: .98 to 1.00)
//     FILTER3           -          1.08        1.05      1.01   1.01   1      1.00
//     FILTER5           -          1.11        1.04      1.01   1.00   1      1.00
//     FILTER_F32        -          1.08        1.03      1.01   1.00   1      1.01
//     BOX              0.99        1.03        1.01      1      1.00   1.00   1.00   (.88 to 1.12, 1.03 to 1.17)
//     DPASD_IJ          -          1.05        0.98      1.00   1      1.00   1.00   (100: .92 to 1.02)
//     DPASD_K          0.90        1.06        1.02      1      0.99   0.99   0.99   (2 a unit: .65 on the small grids)
//     VJP_MARCH        1.16        1.09        1.04      1.01   1      1.00   1.00
//     VJP_FINISH       1.06        1.06        1.00      1      1.00   1.00   1.00
//     FORMT            1.08        1.01        0.99      1      1.00   1.00   1.00
// So slots that fit the kernel matter, and any drift from 500 up serves; they need another look when a
// kernel's registers, LDS or tile change.
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
