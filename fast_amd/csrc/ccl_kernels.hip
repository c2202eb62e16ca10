// gfx950 kernels of the reachable-pore labelling.
//
// The reference labels 6-connected components of "spans" (fastlib/src/cuda/VolumeCCL.cu:86-375):
// scanning each x-row from a `background` previous value, every change of value toggles a
// span open/closed; spans in neighbouring rows that overlap in x are connected; a component's
// label is the minimum span-start linear index, then labels are renumbered 1..K in increasing
// order of that index.  Two in-span voxels adjacent along x always share a span, so the
// components are exactly the 6-connected components of the in-span voxel set, and the
// renumbering orders components by their minimum linear voxel index.
//
// Here: (1) one thread per row computes the span set and points every in-span voxel at its
// span start; (2) a lock-free union-find links rows across y and z, always towards the lower
// index, so each component's root is its minimum index; (3) a deterministic prefix count of
// roots gives every root its rank, i.e. the reference label; (4) every voxel walks to its root.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>

namespace ftc {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kScanThreads = 256;
constexpr int kScanPer = 16;
constexpr int kScanChunk = kScanThreads * kScanPer;

namespace {

__device__ __forceinline__ uint32_t ld(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// An entry as it is or was: any value it has had is an ancestor, and whether it is kNone is fixed.
__device__ __forceinline__ uint32_t early(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Root of x, pointing every other entry on the way at its grandparent.  An entry only ever takes
// an ancestor of its voxel, and one that is not a root never becomes one, so a store that replaces another
// thread's, be it with a higher ancestor, keeps the entry in its component.
__device__ __forceinline__ uint32_t find_halving(uint32_t* P, uint32_t x) {
    for (;;) {
        const uint32_t p = ld(P + x);
        if (p == x) return x;
        const uint32_t g = ld(P + p);
        if (g == p) return p;
        __hip_atomic_store(P + x, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = g;
    }
}

// Ancestor of x reached over entries as the caches hold them.
__device__ __forceinline__ uint32_t find_early(const uint32_t* P, uint32_t x) {
    for (uint32_t p = early(P + x); p != x; p = early(P + x)) x = p;
    return x;
}

__device__ __forceinline__ void merge(uint32_t* P, uint32_t a, uint32_t b) {
    a = find_early(P, a);
    b = find_early(P, b);
    if (a == b) return;   // a common ancestor: linked already
    for (;;) {
        a = find_halving(P, a);
        b = find_halving(P, b);
        if (a == b) return;
        if (a < b) {
            const uint32_t old = atomicMin(P + b, a);
            if (old == b) return;
            b = old;
        } else {
            const uint32_t old = atomicMin(P + a, b);
            if (old == a) return;
            a = old;
        }
    }
}

// Span starts, one wave per x-row in chunks of 64 voxels; the waves stride over the rows, so
// the grid stays within the launch limit however many rows there are.  A voxel is in a span
// when the number of value changes up to it (from `background` before the row) is odd, and
// its span starts at the last change at or before it; both come from a ballot of the change
// flags, with the parity and the last change carried from chunk to chunk.
__global__ __launch_bounds__(256) void k_spans(const uint8_t* __restrict__ mask, uint32_t* __restrict__ P, int nx,
                                               int rows, uint8_t background) {
    const int lane = threadIdx.x & 63;
    const unsigned long long upto = (2ull << lane) - 1ull;   // lanes 0..lane
    for (long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); row < rows; row += (long long)gridDim.x * 4) {
    const long long base = row * nx;
    int prev_last = background;   // value before this chunk
    unsigned parity = 0;          // number of changes before this chunk, mod 2
    uint32_t last_change = kNone; // index of the last change before this chunk
    for (int x0 = 0; x0 < nx; x0 += 64) {
        const int x = x0 + lane;
        const bool in = x < nx;
        const int v = in ? (int)mask[base + x] : 0;
        int pv = __shfl_up(v, 1, 64);
        if (lane == 0) pv = prev_last;
        const unsigned long long changes = __ballot(in && v != pv);
        const unsigned long long mine = changes & upto;
        const bool open = ((parity + (unsigned)__popcll(mine)) & 1u) != 0u;
        const uint32_t start = mine ? (uint32_t)(base + x0 + (63 - __clzll((long long)mine))) : last_change;
        if (in) P[base + x] = open ? start : kNone;
        parity = (parity + (unsigned)__popcll(changes)) & 1u;
        if (changes) last_change = (uint32_t)(base + x0 + (63 - __clzll((long long)changes)));
        prev_last = __shfl(v, 63, 64);
    }
    }
}

// Link every span to the spans it overlaps in the rows at y-1 and z-1.  A voxel whose byte
// equals its x-1 neighbour's lies in the same span as that neighbour (spans change only where
// the value changes), so where neither this row nor the other row changes value between x-1
// and x, the pair of spans was already linked at x-1 and the voxel is skipped.  Where the voxel, its
// neighbours at y-1 and z-1 and the one at both are all in spans, the link to z-1 is left out too: the voxel
// at y-1 is linked to it there, down to the first row of such a run, and both pairs of rows are
// linked across y.
// Bound by the dependent loads of the walks to the roots.  Loads of the first entries and masks in
// flight together, walks over cached entries before coherent ones, and without the links across z that
// others imply: 250 x 233 x 241 ellipsoids 307 -> 258 us, 192^3 182 -> 143 us.
__global__ __launch_bounds__(256) void k_union(const uint8_t* __restrict__ mask, uint32_t* P, int nx, int ny, int nz) {
    const long long n = (long long)nx * ny * nz;
    const long long plane = (long long)nx * ny;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const unsigned row = (unsigned)i / (unsigned)nx;   // labels are 32-bit, so i < 2^32
        const int x = (int)((unsigned)i - row * (unsigned)nx);
        const int z = (int)(row / (unsigned)ny);
        const int y = (int)(row - (unsigned)z * (unsigned)ny);
        const long long iy = y > 0 ? i - nx : i, iz = z > 0 ? i - plane : i;
        const int left = x > 0 ? 1 : 0;
        const uint32_t here = early(P + i), py = early(P + iy), pz = early(P + iz), pyz = early(P + (iz + iy - i));
        const int m0 = mask[i], m1 = mask[i - left], y0 = mask[iy], y1 = mask[iy - left], z0 = mask[iz], z1 = mask[iz - left];
        if (here == kNone) continue;
        const bool same_here = x > 0 && m0 == m1;
        if (y > 0 && py != kNone && !(same_here && y0 == y1)) merge(P, here, py);
        const bool around = y > 0 && py != kNone && pyz != kNone;
        if (z > 0 && pz != kNone && !around && !(same_here && z0 == z1)) merge(P, here, pz);
    }
}

// (A thread that counted 16 elements of its own, 64 bytes apart from lane to lane, took 35 us to count
// and 63 us to label 250 x 233 x 241 voxels; this form 14 and 15 us.)
// Roots before this thread's element, over a block's chunk of kScanChunk elements: a wave takes a
// contiguous part of it, 64 elements at a time, f(i, rank) is called for every root, rank
// counted from the chunk's start.  Returns the chunk's roots.
template <class F>
__device__ __forceinline__ uint32_t chunk_roots(const uint32_t* __restrict__ P, long long n, F f) {
    constexpr int kWaves = kScanThreads / 64, kPart = kScanChunk / kWaves;
    __shared__ uint32_t wtot[kWaves];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long b0 = (long long)blockIdx.x * kScanChunk + (long long)w * kPart + lane;
    unsigned long long m[kPart / 64];
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kPart / 64; ++k) {
        const long long i = b0 + 64 * k;
        m[k] = __ballot(i < n && P[i] == (uint32_t)i);
        c += (uint32_t)__popcll(m[k]);
    }
    if (lane == 0) wtot[w] = c;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (int i = 0; i < kWaves; ++i) {
        if (i < w) before += wtot[i];
        total += wtot[i];
    }
#pragma unroll
    for (int k = 0; k < kPart / 64; ++k) {
        if ((m[k] >> lane) & 1ull) f(b0 + 64 * k, before + (uint32_t)__popcll(m[k] & ((1ull << lane) - 1ull)));
        before += (uint32_t)__popcll(m[k]);
    }
    return total;
}

__global__ __launch_bounds__(kScanThreads) void k_count_roots(const uint32_t* P, long long n, uint32_t* blocksum) {
    const uint32_t total = chunk_roots(P, n, [](long long, uint32_t) {});
    if (threadIdx.x == 0) blocksum[blockIdx.x] = total;
}

// exclusive scan of nb block sums in one block; total number of roots to *total
__global__ __launch_bounds__(1024) void k_scan_blocks(uint32_t* blocksum, int nb, uint32_t* total) {
    __shared__ uint32_t part[16];
    const int per = (nb + 1023) / 1024;
    const int b0 = threadIdx.x * per;
    uint32_t s = 0;
    for (int k = 0; k < per; ++k)
        if (b0 + k < nb) s += blocksum[b0 + k];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = s;   // sum over the wave's lanes up to this one
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(inc, off, 64);
        if (lane >= off) inc += t;
    }
    if (lane == 63) part[w] = inc;
    __syncthreads();
    uint32_t run = inc - s, all = 0;
    for (int i = 0; i < 16; ++i) {
        if (i < w) run += part[i];
        all += part[i];
    }
    if (threadIdx.x == 0) *total = all;
    for (int k = 0; k < per; ++k) {
        if (b0 + k < nb) {
            const uint32_t t = blocksum[b0 + k];
            blocksum[b0 + k] = run;
            run += t;
        }
    }
}

// roots get label = 1 + number of roots before them in linear order
__global__ __launch_bounds__(kScanThreads) void k_assign_roots(const uint32_t* P, long long n, const uint32_t* blockoff,
                                                               uint32_t* L) {
    const uint32_t first = blockoff[blockIdx.x] + 1u;
    (void)chunk_roots(P, n, [&](long long i, uint32_t rank) { L[i] = first + rank; });
}

// Every other voxel takes its root's label (written by the previous kernel, and not here).  Walking here
// instead of flattening the entries in a pass of its own: 75 + 29 -> 79 us at 250 x 233 x 241.
__global__ __launch_bounds__(256) void k_final_labels(const uint32_t* __restrict__ P, long long n, uint32_t* L) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        uint32_t p = P[i];
        if (p == kNone) {
            L[i] = 0;
        } else if (p != (uint32_t)i) {
            for (uint32_t q = P[p]; q != p; q = P[p]) p = q;
            L[i] = L[p];
        }
    }
}

// face table: row f, label l present on face f (Dir order X+,X-,Y+,Y-,Z+,Z-)
__global__ __launch_bounds__(256) void k_face_table(const uint32_t* L, int nx, int ny, int nz, uint8_t* table,
                                                    uint32_t numLabels) {
    const int f = blockIdx.y;
    const int k = f >> 1;
    const int dims[3] = {nx, ny, nz};
    const int fixed = (f & 1) ? 0 : dims[k] - 1;
    const int s0 = (k + 1) % 3, s1 = (k + 2) % 3;
    const long long m = (long long)dims[s0] * dims[s1];
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < m; q += (long long)gridDim.x * blockDim.x) {
        int pos[3];
        pos[k] = fixed;
        pos[s0] = (int)(q % dims[s0]);
        pos[s1] = (int)(q / dims[s0]);
        const uint32_t l = L[(long long)pos[0] + (long long)nx * ((long long)pos[1] + (long long)ny * pos[2])];
        if (l > 0) table[(size_t)f * numLabels + l] = 1;
    }
}

__global__ __launch_bounds__(256) void k_face_all(uint8_t* table, uint32_t numLabels) {
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < numLabels; l += gridDim.x * blockDim.x) {
        uint8_t a = 1;
        for (int f = 0; f < 6; ++f) a &= table[(size_t)f * numLabels + l];
        table[(size_t)6 * numLabels + l] = a;
    }
}

__global__ __launch_bounds__(256) void k_reachable(const uint32_t* L, long long n, const uint8_t* table, uint32_t numLabels,
                                                   int fa, int fb, uint8_t* out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const uint32_t l = L[i];
        out[i] = (table[(size_t)fa * numLabels + l] && table[(size_t)fb * numLabels + l]) ? 255 : 0;
    }
}

// Face bits of every label: bit f set when it touches face f (rows 0..5 of the face table; label 0, the
// background, is on no row), in place of the table's last row.
__global__ __launch_bounds__(256) void k_face_bits(uint8_t* table, uint32_t numLabels) {
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < numLabels; l += gridDim.x * blockDim.x) {
        uint32_t bits = 0;
#pragma unroll
        for (int f = 0; f < 6; ++f) bits |= (uint32_t)(table[(size_t)f * numLabels + l] != 0) << f;
        table[(size_t)6 * numLabels + l] = (uint8_t)bits;
    }
}

// Face bits of every voxel, one byte per voxel for the six boundary-connected volumes of
// generateBoundaryConnectedVolume (VolumeSegmentation.cpp:66-90).  Four voxels per thread (six
// table bytes and a byte store for each voxel took 31 us for 250 x 233 x 241; this form 13 us).
__global__ __launch_bounds__(256) void k_face_codes(const uint32_t* __restrict__ L, long long n,
                                                    const uint8_t* __restrict__ bits, uint8_t* __restrict__ out) {
    for (long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < n; i += (long long)gridDim.x * blockDim.x * 4) {
        if (i + 4 <= n) {   // both buffers start at an allocation's alignment
            const uint4 l = *reinterpret_cast<const uint4*>(L + i);
            *reinterpret_cast<uint32_t*>(out + i) = (uint32_t)bits[l.x] | (uint32_t)bits[l.y] << 8 |
                                                    (uint32_t)bits[l.z] << 16 | (uint32_t)bits[l.w] << 24;
        } else {
            for (long long j = i; j < n; ++j) out[j] = bits[L[j]];
        }
    }
}

// Per-label statistics (getCCLSegmentInfo, VolumeSegmentation.cpp:135-178): voxel count and
// bounding box.  info[7 l ..]: count, min x, y, z, max x, y, z (inclusive).  Every x-run of
// equal labels contributes once, from its first voxel, with integer atomics (the result does
// not depend on their order).
__global__ __launch_bounds__(256) void k_seg_init(uint32_t* info, uint32_t numLabels, int nx, int ny, int nz) {
    for (long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x; l < numLabels;
         l += (long long)gridDim.x * blockDim.x) {
        uint32_t* r = info + 7 * l;
        r[0] = 0;
        r[1] = (uint32_t)nx;
        r[2] = (uint32_t)ny;
        r[3] = (uint32_t)nz;
        r[4] = r[5] = r[6] = 0;
    }
}

__global__ __launch_bounds__(256) void k_seg_runs(const uint32_t* L, int nx, int ny, int nz, uint32_t* info) {
    const long long n = (long long)nx * ny * nz;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const uint32_t l = L[i];
        const unsigned row = (unsigned)i / (unsigned)nx;
        const int x = (int)((unsigned)i - row * (unsigned)nx);
        if (x > 0 && L[i - 1] == l) continue;   // not the first voxel of its run
        int e = x;
        while (e + 1 < nx && L[i + (e + 1 - x)] == l) ++e;
        const int y = (int)(row % (unsigned)ny);
        const int z = (int)(row / (unsigned)ny);
        uint32_t* r = info + 7 * (size_t)l;
        atomicAdd(r + 0, (uint32_t)(e - x + 1));
        atomicMin(r + 1, (uint32_t)x);
        atomicMin(r + 2, (uint32_t)y);
        atomicMin(r + 3, (uint32_t)z);
        atomicMax(r + 4, (uint32_t)e);
        atomicMax(r + 5, (uint32_t)y);
        atomicMax(r + 6, (uint32_t)z);
    }
}

inline unsigned grid_for(long long n) {
    long long b = (n + 255) / 256;
    return (unsigned)(b > 65536 ? 65536 : (b < 1 ? 1 : b));
}

}  // namespace

// Labels (0 = background, 1..K canonical) into L; returns K via *num_roots (device, 1 uint32).
// P, L: n uint32 each; blocksum: ceil(n / 4096) uint32.
hipError_t ccl_label(const uint8_t* mask, int nx, int ny, int nz, uint8_t background, uint32_t* P, uint32_t* L,
                     uint32_t* blocksum, uint32_t* num_roots, hipStream_t s) {
    const long long n = (long long)nx * ny * nz;
    const int rows = ny * nz;   // < 2^31: volumes hold fewer than 2^31 voxels
    const int span_blocks = std::min((rows + 3) / 4, 65536);   // 4 rows per block and sweep
    hipLaunchKernelGGL(k_spans, dim3(span_blocks), dim3(256), 0, s, mask, P, nx, rows, background);
    hipLaunchKernelGGL(k_union, dim3(grid_for(n)), dim3(256), 0, s, mask, P, nx, ny, nz);
    const int nb = (int)((n + kScanChunk - 1) / kScanChunk);
    hipLaunchKernelGGL(k_count_roots, dim3(nb), dim3(kScanThreads), 0, s, (const uint32_t*)P, n, blocksum);
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, blocksum, nb, num_roots);
    hipLaunchKernelGGL(k_assign_roots, dim3(nb), dim3(kScanThreads), 0, s, (const uint32_t*)P, n,
                       (const uint32_t*)blocksum, L);
    hipLaunchKernelGGL(k_final_labels, dim3(grid_for(n)), dim3(256), 0, s, (const uint32_t*)P, n, L);
    return hipGetLastError();
}

// 7 x numLabels face table (must be zeroed by the caller).
hipError_t ccl_face_table(const uint32_t* L, int nx, int ny, int nz, uint8_t* table, uint32_t numLabels, hipStream_t s) {
    const long long maxface = (long long)std::max(nx, ny) * std::max(std::max(ny, nz), nx) + (long long)nz * nx;
    hipLaunchKernelGGL(k_face_table, dim3(grid_for(maxface), 6), dim3(256), 0, s, L, nx, ny, nz, table, numLabels);
    hipLaunchKernelGGL(k_face_all, dim3(grid_for(numLabels)), dim3(256), 0, s, table, numLabels);
    return hipGetLastError();
}

hipError_t ccl_reachable(const uint32_t* L, long long n, const uint8_t* table, uint32_t numLabels, int dir, uint8_t* out,
                         hipStream_t s) {
    const int k = dir / 2;
    hipLaunchKernelGGL(k_reachable, dim3(grid_for(n)), dim3(256), 0, s, L, n, table, numLabels, 2 * k, 2 * k + 1, out);
    return hipGetLastError();
}

hipError_t ccl_segment_stats(const uint32_t* L, int nx, int ny, int nz, uint32_t numLabels, uint32_t* info,
                             hipStream_t s) {
    const long long n = (long long)nx * ny * nz;
    hipLaunchKernelGGL(k_seg_init, dim3(grid_for(numLabels)), dim3(256), 0, s, info, numLabels, nx, ny, nz);
    hipLaunchKernelGGL(k_seg_runs, dim3(grid_for(n)), dim3(256), 0, s, L, nx, ny, nz, info);
    return hipGetLastError();
}

// table: the 7 x numLabels face table; its last row is overwritten.
hipError_t ccl_face_codes(const uint32_t* L, long long n, uint8_t* table, uint32_t numLabels, uint8_t* out, hipStream_t s) {
    hipLaunchKernelGGL(k_face_bits, dim3(grid_for(numLabels)), dim3(256), 0, s, table, numLabels);
    hipLaunchKernelGGL(k_face_codes, dim3(grid_for((n + 3) / 4)), dim3(256), 0, s, L, n, (const uint8_t*)table + (size_t)6 * numLabels, out);
    return hipGetLastError();
}

}  // namespace ftc
