// Rows gathered through LDS: how a wavefront reads the cell and gradient rows of 64 other cells (the sweep's neighbours, a
// face kernel's far sides) in whole lines. For kernels of one wavefront per work-group.
#pragma once

#include "kernels.hpp"

namespace luna {

template <int D>
__device__ __forceinline__ void load_vec(const double* p, double* v) {
#pragma unroll
    for (int a = 0; a < D; ++a) v[a] = p[a];
}

// One list entry as the sweep's first walk reads it: the face's |A| (from the entry's slot) and the other cell's row.
template <int D>
struct Near {
    double mag, x[D], c[D], W[D + 2], cs;
};

typedef __attribute__((address_space(3))) double lds_double;
typedef double double2v __attribute__((ext_vector_type(2)));

// A work-group's staged rows in LDS. They are filled and read 16 B at a time, which a plain array of doubles does not promise
// the alignment of (another __shared__ variable before it may leave it at 8).
template <int DOUBLES>
struct alignas(16) StagedRows {
    double at[DOUBLES];
    static_assert(DOUBLES % 2 == 0, "whole 16 B chunks");

    __device__ __forceinline__ lds_double* lds() { return (lds_double*)at; }
};
static_assert(alignof(StagedRows<2>) == sizeof(double2v), "ds_read_b128 and the 16 B loads to LDS");

// A wavefront's neighbour rows through LDS. A lane that loads its own neighbour's row itself touches a 128 B line per 16 B
// load, and a CU's L1 looks up one line a cycle: the rows of 64 neighbours cost 7 x 64 lookups, which bound the list walk
// (5.6 thousand cycles an entry at 12 wavefronts a CU). Here the 16 B chunks of all 64 rows are dealt to the lanes in order
// (chunk q to lane q mod 64 of load q / 64, of row q / CHUNKS), so that a load covers whole rows, and go to LDS without
// passing through registers, back to back (a row at 16 CHUNKS bytes times its lane). Chunks with neither x, c, W nor c_s
// (V and r) are skipped. Two buffers: one is read while the other is in flight.
template <int D>
struct Stage {
    static constexpr int CHUNKS = D == 3 ? 6 : 5, ROW = 2 * CHUNKS;  // a staged row: [x, c, W, c_s]
    static constexpr int DOUBLES = 2 * 64 * ROW;                      // both buffers
    static constexpr int SKIP = D;                                    // staged chunks before it are a row's first, the others its from GEO_ROW / 2 on
    static constexpr int PERIOD = D == 3 ? 3 : 5;                     // load k + PERIOD takes the same chunks of rows 32 further (3D)
    int from[PERIOD], chunk[PERIOD];  // per load: 4 x the lane whose neighbour this lane fetches for, the chunk of its row
    unsigned at[CHUNKS];              // per load: the next fetch's source, in chunks from the first cell row
    lds_double* buffer;
    unsigned row;  // the LDS address of this lane's row in buffer 0

    __device__ __forceinline__ void init(int lane, lds_double* lds) {
#pragma unroll
        for (int k = 0; k < PERIOD; ++k) {
            const int q = k * 64 + lane, c = q % CHUNKS;
            from[k] = q / CHUNKS * 4;
            chunk[k] = c < SKIP ? c : c - SKIP + GEO_ROW / 2;
        }
        buffer = lds;
        row = (unsigned)(size_t)lds + lane * ROW * 8;
    }
    // The sources of a fetch of the cells j's rows (one a lane; every lane active).
    __device__ __forceinline__ void address(int j) {
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k)
            at[k] = (unsigned)__builtin_amdgcn_ds_bpermute(from[k % PERIOD] + k / PERIOD * 128, j) << 3 | (unsigned)chunk[k % PERIOD];
    }
    __device__ __forceinline__ void fetch(const double* cell, int b) const {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            const char* src = reinterpret_cast<const char*>(cell) + (size_t)at[k] * 16;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)(buffer + b * (64 * ROW) + k * 128), 16, 0, 0);
        }
        asm volatile("" ::: "memory");
    }
    // This lane's row in buffer b, whose fetch may be followed by one other of CHUNKS loads that is still in flight. The reads
    // are complete when this returns, so that the next fetch may overwrite the buffer.
    __device__ __forceinline__ void read(int b, Near<D>& n) const {
        const unsigned p = row + b * (64 * ROW * 8);
        double2v d[CHUNKS];
        if constexpr (D == 3)
            asm volatile(
                "s_waitcnt vmcnt(6)\n\tds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:16\n\tds_read_b128 %2, %6 offset:32\n\t"
                "ds_read_b128 %3, %6 offset:48\n\tds_read_b128 %4, %6 offset:64\n\tds_read_b128 %5, %6 offset:80\n\ts_waitcnt lgkmcnt(0)"
                : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3]), "=&v"(d[4]), "=&v"(d[CHUNKS - 1])
                : "v"(p)
                : "memory");
        else
            asm volatile(
                "s_waitcnt vmcnt(5)\n\tds_read_b128 %0, %5\n\tds_read_b128 %1, %5 offset:16\n\tds_read_b128 %2, %5 offset:32\n\t"
                "ds_read_b128 %3, %5 offset:48\n\tds_read_b128 %4, %5 offset:64\n\ts_waitcnt lgkmcnt(0)"
                : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3]), "=&v"(d[4])
                : "v"(p)
                : "memory");
        const auto v = [&](int k) { return k & 1 ? d[k / 2].y : d[k / 2].x; };
#pragma unroll
        for (int a = 0; a < D; ++a) {
            n.x[a] = v(a);
            n.c[a] = v(D + a);
        }
#pragma unroll
        for (int w = 0; w < D + 2; ++w) n.W[w] = v(2 * D + w);
        n.cs = v(3 * D + 2);
    }
    // Nothing in flight to LDS any more.
    __device__ __forceinline__ void drain() const { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
};

// One side of a face, from its cell's rows in memory. A gradient row of Prec: 16 B chunks GradientRow::CHUNKS.
template <int D, int Prec>
struct GradientRow {
    static constexpr int CHUNKS = (Prec == 0 ? grad_row<D>() * 8 : Prec == 1 ? lp_row<D>() * 4 : HALF_ROW * 2) / 16;
};
template <int D, int Prec>
struct MemorySide {
    const double* row;
    const double2v* grad;
    __device__ __forceinline__ MemorySide(const Geo& g, const Rows& r, int i)
        : row(g.cell + (size_t)i * CELL_ROW), grad(reinterpret_cast<const double2v*>(r.grad) + (size_t)i * GradientRow<D, Prec>::CHUNKS) {}
    __device__ __forceinline__ void place(double* x, double* c) const {
        using C = CellAt<D>;
        load_vec<D>(row + C::X, x);
        load_vec<D>(row + C::C, c);
    }
    __device__ __forceinline__ void state(double* W) const {
#pragma unroll
        for (int v = 0; v < D + 2; ++v) W[v] = row[CellAt<D>::W + v];
    }
    __device__ __forceinline__ double2v chunk(int k) const { return grad[k]; }
};

// The same from LDS, where a wavefront's 64 neighbours' rows are fetched in whole lines (as the sweep's Stage, whose reason
// holds here: 14 loads a side of which each lane's touches a line of its own kept the L1's lookups at 85 % and the address
// unit at 97 % of the flux kernel's time). The state part of a cell row is laid out as Stage does it; a gradient row keeps
// its chunks together, chunk c of row l at place c ^ (l mod CHUNKS), so that lanes reading the same chunk of their rows
// read different banks.
template <int D, int Prec>
struct StagedSide {
    static constexpr int CELL = Stage<D>::CHUNKS, GRAD = GradientRow<D, Prec>::CHUNKS;
    static constexpr int DOUBLES = 64 * 2 * (CELL + GRAD);
    const lds_double* cell;
    const lds_double* grad;
    int lane;
    __device__ __forceinline__ StagedSide(lds_double* lds, int lane) : cell(lds + lane * 2 * CELL), grad(lds + 64 * 2 * CELL + lane * 2 * GRAD), lane(lane) {}
    // The rows of the cells j (one a lane; every lane of the wavefront active), asynchronously: finish() before reading.
    static __device__ __forceinline__ void fetch(const Geo& g, const Rows& r, int j, bool gradients, lds_double* lds, int lane) {
#pragma unroll
        for (int k = 0; k < CELL; ++k) {
            const int q = k * 64 + lane, c = q % CELL;
            const unsigned of = (unsigned)__builtin_amdgcn_ds_bpermute(q / CELL * 4, j);
            load(g.cell, (size_t)(of << 3 | (unsigned)(c < D ? c : c - D + GEO_ROW / 2)), lds + k * 128);
        }
        if (gradients) fetch_gradients(r.grad, j, lds + 64 * 2 * CELL, lane);
    }
    static __device__ __forceinline__ void fetch_gradients(const double* from, int j, lds_double* lds, int lane) {
#pragma unroll
        for (int k = 0; k < GRAD; ++k) {
            const int row = k * (64 / GRAD) + lane / GRAD;
            const unsigned of = (unsigned)__builtin_amdgcn_ds_bpermute(row * 4, j);
            load(from, (size_t)of * GRAD + ((lane ^ row) & (GRAD - 1)), lds + k * 128);
        }
    }
    static __device__ __forceinline__ void load(const double* from, size_t chunk, lds_double* to) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(reinterpret_cast<const char*>(from) + chunk * 16),
                                         (__attribute__((address_space(3))) void*)to, 16, 0, 0);
    }
    static __device__ __forceinline__ void finish() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
    __device__ __forceinline__ void place(double* x, double* c) const {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            x[a] = cell[a];
            c[a] = cell[D + a];
        }
    }
    __device__ __forceinline__ void state(double* W) const {
#pragma unroll
        for (int v = 0; v < D + 2; ++v) W[v] = cell[2 * D + v];
    }
    __device__ __forceinline__ double2v chunk(int k) const { return at(grad, lane, k); }
    // Chunk k of this lane's row among the gradient rows that fetch_gradients put at lds.
    static __device__ __forceinline__ double2v gradient_chunk(const lds_double* lds, int lane, int k) { return at(lds + lane * 2 * GRAD, lane, k); }
    static __device__ __forceinline__ double2v at(const lds_double* row, int lane, int k) {
        return *reinterpret_cast<const __attribute__((address_space(3))) double2v*>(row + 2 * (k ^ (lane & (GRAD - 1))));
    }
};
template <int D, class S>
__device__ __forceinline__ void load_gradient(const S& side, double* gr) {
#pragma unroll
    for (int k = 0; k < (D + 2) * D; k += 2) {
        const double2v d = side.chunk(k / 2);
        gr[k] = d.x;
        if (k + 1 < (D + 2) * D) gr[k + 1] = d.y;
    }
}

}  // namespace luna
