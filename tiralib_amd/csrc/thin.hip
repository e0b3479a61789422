// thin.hip -- the consumer end of tensor voting on gfx950: stick saliency,
// Otsu threshold and Lee's 3D thinning.
//
//   * 2D stick saliency |l|max - |l|min (reconstruct.py:14-34); the 3D
//     magnitude-ranked saliency is an eig3 output mode (TIRA_EIG_MAGNITUDE);
//   * Otsu's threshold over a 256-bin histogram on [0, max]
//     (reconstruct.py:37-63) with numpy.histogram's float32 binning rules,
//     all on the device (max reduction, LDS-privatised histogram, one-thread
//     scan in FP64), then the binary mask `s > t`;
//   * Lee et al. 1994 thinning as tira::lee / computeThinImage implement it
//     (thinning/lee_thinning.h:600-706), bit-exact. Per border direction the
//     reference collects candidates on the unchanged volume, then re-checks
//     them one by one in raster order, so a candidate sees the deletions of
//     the candidates before it. Here candidates are collected in parallel and
//     the sequential re-check is solved as the fixed point of
//       keep(p) = not simple(N_p with earlier deleted candidates removed),
//     iterated in parallel (Jacobi) until no decision changes: the decisions
//     form a DAG along raster order, whose solution is unique, so any fixed
//     point is the sequential result.
// Neighbourhoods are 27-bit codes, bit 9(dz+1) + 3(dy+1) + (dx+1), the order
// of get_neighborhood (lee_thinning.h:52-91); bit 13 is the voxel itself.
#include "common.hpp"
#include "eig_device.hpp"

#include <vector>

namespace th {

// ---------------------------------------------------------------- neighbourhood tests
// Bits with x = 0 / x = 2 / y = 0 / y = 2 inside the 3x3x3 code.
constexpr unsigned kX0 = 0x1249249u, kX2 = 0x4924924u, kY0 = 0x01C0E07u, kY2 = 0x70381C0u, kAll = 0x7FFFFFFu;

// 3x3x3 dilation of a set of neighbourhood bits, one axis at a time; each
// step is clipped to the 27 bits, or a left shift past bit 26 would come back
// into range with the next right shift.
TH_HD inline unsigned dilate26(unsigned s) {
    s = (s | ((s << 1) & ~kX0) | ((s >> 1) & ~kX2)) & kAll;
    s = (s | ((s << 3) & ~kY0) | ((s >> 3) & ~kY2)) & kAll;
    return (s | (s << 9) | (s >> 9)) & kAll;
}

// Simple-point test of is_simple_point (lee_thinning.h:530-579): the 26
// neighbours form at most one 26-connected component. Flood fill by repeated
// 3x3x3 dilation inside the neighbour set.
TH_HD inline bool thin_simple(unsigned code) {
    const unsigned obj = code & ~(1u << 13) & kAll;
    if (!obj) return true;
    unsigned c = obj & (0u - obj);
    for (;;) {
        const unsigned g = dilate26(c) & obj;
        if (g == c) break;
        c = g;
    }
    return c == obj;
}

// Mask of the voxels other than the centre that share the centre cube's cell
// (sx, sy, sz): s = 0 spans an axis, +-1 lies on that side (a vertex has
// three nonzero s, an edge two, a face one).
TH_HD constexpr unsigned cell_mask(int sx, int sy, int sz) {
    unsigned m = 0;
    for (int ox = (sx < 0 ? sx : 0); ox <= (sx > 0 ? sx : 0); ox++)
        for (int oy = (sy < 0 ? sy : 0); oy <= (sy > 0 ? sy : 0); oy++)
            for (int oz = (sz < 0 ? sz : 0); oz <= (sz > 0 ? sz : 0); oz++)
                if (ox || oy || oz) m |= 1u << (9 * (oz + 1) + 3 * (oy + 1) + (ox + 1));
    return m;
}

// Euler invariance of is_euler_invariant (lee_thinning.h:288-299), computed as
// the change of V - E + F - C of the union of closed voxel cubes when the
// centre cube is removed: only centre-cube cells that no other voxel's cube
// contains disappear. Equivalent to the octant-LUT sum being zero over all
// 2^26 neighbourhoods.
TH_HD inline bool thin_euler_invariant(unsigned code) {
    int d = -1;
#pragma unroll
    for (int sx = -1; sx <= 1; sx++)
#pragma unroll
        for (int sy = -1; sy <= 1; sy++)
#pragma unroll
            for (int sz = -1; sz <= 1; sz++) {
                const int dim = (sx == 0) + (sy == 0) + (sz == 0);
                if (dim == 3) continue;
                if ((code & cell_mask(sx, sy, sz)) == 0) d += (dim % 2 == 0) ? 1 : -1;
            }
    return d == 0;
}

// is_endpoint (lee_thinning.h:96-103): exactly one set neighbour.
TH_HD inline bool thin_endpoint(unsigned code) { return __builtin_popcount(code) == 2; }

// Code of voxel (x, y, z) in a 0/1 byte volume (s2 = x fastest), zero outside.
__device__ __forceinline__ unsigned thin_code(const unsigned char* __restrict__ v, int s0, int s1, int s2, int x,
                                              int y, int z) {
    unsigned code = 0;
#pragma unroll
    for (int dz = -1; dz <= 1; dz++) {
        const int Z = z + dz;
        if ((unsigned)Z >= (unsigned)s0) continue;
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            const int Y = y + dy;
            if ((unsigned)Y >= (unsigned)s1) continue;
            const unsigned char* row = v + ((size_t)Z * s1 + Y) * s2;
#pragma unroll
            for (int dx = -1; dx <= 1; dx++) {
                const int X = x + dx;
                if ((unsigned)X < (unsigned)s2 && row[X] == 1) code |= 1u << (9 * (dz + 1) + 3 * (dy + 1) + dx + 1);
            }
        }
    }
    return code;
}

// The same code of a voxel one or more in from every face: nine 4-byte loads
// (three voxels of a row each; the fourth byte stays inside the volume's n
// bytes) instead of 27 byte loads with their bounds. The bytes are 0 or 1.
__device__ __forceinline__ unsigned thin_code_inner(const unsigned char* __restrict__ v, int s1, int s2, size_t i) {
    unsigned code = 0;
#pragma unroll
    for (int dz = -1; dz <= 1; dz++)
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            unsigned w;
            __builtin_memcpy(&w, v + (i + (long long)(dz * s1 + dy) * s2 - 1), 4);
            const unsigned b = (w & 1u) | ((w >> 7) & 2u) | ((w >> 14) & 4u);
            code |= b << (9 * (dz + 1) + 3 * (dy + 1));
        }
    return code;
}

// Appends the `take` threads' values (and second values, list2 not NULL) of a
// block of 256 to list[*count ..]: one atomic per block. Every thread of the
// block calls it, the same number of times.
__device__ __forceinline__ void block_append(bool take, unsigned value, unsigned value2, unsigned* __restrict__ list,
                                             unsigned* __restrict__ list2, unsigned* __restrict__ count) {
    __shared__ unsigned s_cnt[4], s_base;
    const unsigned long long m = __ballot(take);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) s_cnt[wave] = (unsigned)__popcll(m);
    __syncthreads();
    const unsigned c0 = s_cnt[0], c1 = s_cnt[1], c2 = s_cnt[2], total = c0 + c1 + c2 + s_cnt[3];
    if (threadIdx.x == 0 && total) s_base = atomicAdd(count, total);
    __syncthreads();
    if (take) {
        const unsigned slot = s_base + (wave > 0 ? c0 : 0u) + (wave > 1 ? c1 : 0u) + (wave > 2 ? c2 : 0u) +
                              (unsigned)__popcll(m & ((1ull << lane) - 1ull));
        list[slot] = value;
        if (list2) list2[slot] = value2;
    }
    __syncthreads();  // the next call writes s_cnt and s_base
}

// Raises *flag if any lane hit. A flag and no count: hits of thousands of
// waves on one counter queue up, equal stores do not.
__device__ __forceinline__ void wave_flag(bool hit, unsigned* __restrict__ flag) {
    const unsigned long long m = __ballot(hit);
    if (m && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)m) - 1)) *flag = 1u;
}

// ---------------------------------------------------------------- thinning kernels
// Binarise (lee(), lee_thinning.h:690-699): any nonzero value becomes 1.
template <typename T>
__global__ __launch_bounds__(256) void k_thin_binarise(const T* in, unsigned char* v, size_t n) {  // may alias
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        v[i] = in[i] != (T)0 ? 1 : 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_thin_export(const unsigned char* __restrict__ v, T* __restrict__ out,
                                                     size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = (T)v[i];
}

// Object voxels (value 1) among the nfrom listed ones (from NULL: of the whole
// volume, nfrom = n) appended to `list` (NULL: counted); every thread runs the
// same number of iterations. stall (optional): see k_thin_apply.
__global__ __launch_bounds__(256) void k_thin_objects(const unsigned char* __restrict__ v,
                                                      const unsigned* __restrict__ from, size_t nfrom,
                                                      unsigned* __restrict__ list, unsigned* __restrict__ count,
                                                      const unsigned* __restrict__ stall) {
    if (stall && *stall) return;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t iters = (nfrom + stride - 1) / stride;
    for (size_t it = 0; it < iters; it++) {
        const size_t k = it * stride + (size_t)blockIdx.x * blockDim.x + threadIdx.x;
        unsigned i = 0;
        bool take = false;
        if (k < nfrom) {
            i = from ? from[k] : (unsigned)k;
            take = v[i] == 1;
        }
        if (list) {
            block_append(take, i, 0u, list, nullptr, count);
        } else {
            const unsigned long long m = __ballot(take);
            if (m && (threadIdx.x & 63) == 0) atomicAdd(count, (unsigned)__popcll(m));
        }
    }
}

// The object voxels of a volume of 0 / 1 bytes (16-byte aligned): block b takes
// the `per` bytes from b * per (a multiple of 4096), counts them, reserves its
// part of the list with one atomic, reads them again and writes their indices.
// list NULL: the count only. One atomic per wave and a byte per lane took 170 us
// a pass over 12.6 M voxels, this 15 us.
__global__ __launch_bounds__(256) void k_thin_objects_vol(const unsigned char* __restrict__ v, size_t n, size_t per,
                                                          unsigned* __restrict__ list,
                                                          unsigned* __restrict__ count) {
    __shared__ unsigned s_wave[4], s_base;
    const size_t lo = (size_t)blockIdx.x * per, hi = min(n, lo + per);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // the set bytes of 16 voxels from i on, as four words of 0 / 1 bytes
    auto words = [&](size_t i) {
        uint4 w = make_uint4(0, 0, 0, 0);
        if (i + 16 <= hi) w = *reinterpret_cast<const uint4*>(v + i);
        else
            for (int b = 0; b < 16 && i + b < hi; b++)
                (&w.x)[b >> 2] |= (unsigned)v[i + b] << (8 * (b & 3));
        return make_uint4(w.x & 0x01010101u, w.y & 0x01010101u, w.z & 0x01010101u, w.w & 0x01010101u);
    };
    auto ones = [](const uint4& w) { return __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w); };
    unsigned c = 0;
    for (size_t i = lo + threadIdx.x * 16; i < hi; i += 4096) c += (unsigned)ones(words(i));
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor((int)c, d);
    if (lane == 0) s_wave[wave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned t = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        s_base = t ? atomicAdd(count, t) : 0u;
    }
    if (!list) return;
    __syncthreads();
    unsigned base = s_base;
    for (size_t i0 = lo; i0 < hi; i0 += 4096) {  // the same trips for every thread of the block
        const size_t i = i0 + threadIdx.x * 16;
        const uint4 w = words(i);
        const unsigned mine = (unsigned)ones(w);
        unsigned inc = mine;
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned o = (unsigned)__shfl_up((int)inc, d);
            if (lane >= d) inc += o;
        }
        __syncthreads();  // the previous trip's sums are read
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        unsigned at = base + inc - mine;
        for (int k = 0; k < wave; k++) at += s_wave[k];
        base += s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        for (int k = 0; k < 4; k++)
            for (unsigned m = (&w.x)[k]; m; m &= m - 1)
                list[at++] = (unsigned)(i + 4 * k + (__builtin_ctz(m) >> 3));
    }
}

// Candidates of border direction `dir` (0..5 = N y-1, S y+1, E x+1, W x-1,
// U z+1, B z-1; lee_thinning.h:142-147, 623-628) among the listed object
// voxels: voxels whose neighbour in that direction is 0 (or outside), that are
// not end points, are Euler invariant and simple (lee_thinning.h:614-646).
// Each candidate's 26-neighbourhood code goes to codes[] beside its index:
// the volume does not change until the direction's deletions are applied, so
// the re-check sweeps read it instead of the 26 neighbours.
__global__ __launch_bounds__(256) void k_thin_candidates_list(const unsigned char* __restrict__ v, int s0, int s1,
                                                              int s2, int dir, const unsigned* __restrict__ obj,
                                                              unsigned nobj, unsigned char* __restrict__ mark,
                                                              unsigned* __restrict__ list,
                                                              unsigned* __restrict__ codes,
                                                              unsigned* __restrict__ count,
                                                              const unsigned* __restrict__ stall) {
    if (*stall) return;
    const size_t n = (size_t)s0 * s1 * s2;
    const int ddx = dir == 2 ? 1 : dir == 3 ? -1 : 0;
    const int ddy = dir == 0 ? -1 : dir == 1 ? 1 : 0;
    const int ddz = dir == 4 ? 1 : dir == 5 ? -1 : 0;
    const unsigned stride = gridDim.x * blockDim.x;
    const unsigned iters = (nobj + stride - 1) / stride;
    for (unsigned it = 0; it < iters; it++) {
        const unsigned k = it * stride + blockIdx.x * blockDim.x + threadIdx.x;
        bool take = false;
        unsigned i = 0, code = 0;
        if (k < nobj) {
            i = obj[k];
            if (v[i] == 1) {
                const int x = (int)(i % (unsigned)s2), y = (int)((i / (unsigned)s2) % (unsigned)s1);
                const int z = (int)(i / ((unsigned)s1 * (unsigned)s2));
                const int X = x + ddx, Y = y + ddy, Z = z + ddz;
                const bool border = (unsigned)X >= (unsigned)s2 || (unsigned)Y >= (unsigned)s1 ||
                                    (unsigned)Z >= (unsigned)s0 || v[((size_t)Z * s1 + Y) * s2 + X] == 0;
                if (border) {
                    // the last of the inner form's reads is 2 past the farthest neighbour row's middle
                    const bool inner = x > 0 && x + 1 < s2 && y > 0 && y + 1 < s1 && z > 0 && z + 1 < s0 &&
                                       (size_t)i + ((size_t)s1 + 1) * s2 + 2 < n;
                    code = inner ? thin_code_inner(v, s1, s2, i) : thin_code(v, s0, s1, s2, x, y, z);
                    take = !thin_endpoint(code) && thin_euler_invariant(code) && thin_simple(code);
                }
            }
        }
        if (take) mark[i] = 1;
        block_append(take, i, code, list, codes, count);
    }
}

// The sequential re-check (lee_thinning.h:651-661) as a relaxation in place:
// candidate p is deleted (mark 1) when it is simple in the volume where the
// candidates before it in raster order (neighbour bits 0..12) that are
// currently marked for deletion are removed; otherwise kept (mark 2). A
// decision depends on earlier candidates only, so whatever the order of the
// updates the marks settle, level by level, on the one solution; a launch that
// changes no mark has verified it. `rounds` re-evaluations per launch: the
// marks other waves wrote meanwhile are seen where the caches show them, and a
// candidate without earlier candidates around it is done after the first.
// The candidate count is read from device memory (the candidate pass wrote
// it), so the host launches over an upper bound without reading it back.
// codes[k]: candidate k's neighbourhood code (k_thin_candidates_list); a set
// bit is an object neighbour, inside the volume, so its index is the
// candidate's plus the bit's offset.
// changes: raised if a mark changed. prev (optional): that of the previous launch; zero means the marks
// are settled, and the launch returns at once.
__global__ __launch_bounds__(256) void k_thin_resolve(int s1, int s2, const unsigned* __restrict__ list,
                                                      const unsigned* __restrict__ codes,
                                                      const unsigned* __restrict__ count,
                                                      unsigned char* mark, unsigned* __restrict__ changes,
                                                      const unsigned* __restrict__ prev, int rounds) {
    if (prev && *prev == 0u) return;
    const unsigned cnt = *count;
    const unsigned stride = gridDim.x * blockDim.x;
    const unsigned iters = (cnt + stride - 1) / stride;
    const long long plane = (long long)s1 * s2;
    for (unsigned it = 0; it < iters; it++) {
        const unsigned k = it * stride + blockIdx.x * blockDim.x + threadIdx.x;
        bool changed = false;
        if (k < cnt) {
            const size_t i = list[k];
            const unsigned code = codes[k];
            unsigned near = code & 0x1FFFu;  // earlier neighbours; from the second round on, candidates only
            unsigned char own = __hip_atomic_load(mark + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (int round = 0; round < rounds; round++) {
                unsigned c = code, todo = near;
                while (todo) {
                    const int b = __builtin_ctz(todo);
                    todo &= todo - 1;
                    const int dx = b % 3 - 1, dy = (b / 3) % 3 - 1, dz = b / 9 - 1;
                    const size_t q = (size_t)((long long)i + dz * plane + (long long)dy * s2 + dx);
                    const unsigned char m = __hip_atomic_load(mark + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (m == 0) near &= ~(1u << b);
                    if (m == 1) c &= ~(1u << b);
                }
                const unsigned char m = thin_simple(c) ? 1 : 2;
                if (m != own) {
                    __hip_atomic_store(mark + i, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    own = m;
                    changed = true;
                }
                if (!near) break;
            }
        }
        wave_flag(changed, changes);
    }
}

// Apply the decisions: delete marked candidates (deleted: raised if there is
// one), clear the marks. unsettled (optional): whether the last re-check changed
// a mark; if so nothing is
// applied and *stall becomes `tag`, on which the pass's later launches do
// nothing, and the host takes this direction up again.
__global__ __launch_bounds__(256) void k_thin_apply(unsigned char* __restrict__ v, const unsigned* __restrict__ list,
                                                    const unsigned* __restrict__ count,
                                                    unsigned char* __restrict__ mark,
                                                    unsigned* __restrict__ deleted,
                                                    const unsigned* __restrict__ unsettled,
                                                    unsigned* __restrict__ stall, unsigned tag) {
    if (unsettled && *unsettled) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *stall = tag;
        return;
    }
    const unsigned cnt = *count;
    const unsigned stride = gridDim.x * blockDim.x;
    const unsigned iters = (cnt + stride - 1) / stride;
    for (unsigned it = 0; it < iters; it++) {
        const unsigned k = it * stride + blockIdx.x * blockDim.x + threadIdx.x;
        bool del = false;
        if (k < cnt) {
            const size_t i = list[k];
            del = mark[i] == 1;
            if (del) v[i] = 0;
            mark[i] = 0;
        }
        wave_flag(del, deleted);
    }
}

// Per-code flags of the three tests (bit 0 Euler invariant, bit 1 simple,
// bit 2 end point) for codes `first + k` enumerated with the centre set:
// code = low 13 bits | 1 << 13 | high bits << 14.
__global__ __launch_bounds__(256) void k_thin_classify(unsigned first, unsigned count,
                                                       unsigned char* __restrict__ flags) {
    for (unsigned k = blockIdx.x * blockDim.x + threadIdx.x; k < count; k += gridDim.x * blockDim.x) {
        const unsigned e = first + k;
        const unsigned code = (e & 0x1FFFu) | (1u << 13) | ((e >> 13) << 14);
        flags[k] = (unsigned char)((thin_euler_invariant(code) ? 1 : 0) | (thin_simple(code) ? 2 : 0) |
                                   (thin_endpoint(code) ? 4 : 0));
    }
}

__global__ __launch_bounds__(256) void k_thin_zero_n(unsigned* __restrict__ c, int n) {
    for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) c[i] = 0u;
}

__global__ void k_thin_zero(unsigned* __restrict__ c, int n) {
    if ((int)threadIdx.x < n) c[threadIdx.x] = 0u;
}

__global__ __launch_bounds__(256) void k_fill_u8(unsigned char* __restrict__ p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0;
}

__global__ void k_fill_u64(unsigned long long* __restrict__ p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// ---------------------------------------------------------------- saliency and Otsu
// 2D stick saliency |l|max - |l|min of [a b; b c] (reconstruct.py:14-34).
__global__ __launch_bounds__(256) void k_stick_saliency2(const float4* __restrict__ t, size_t n,
                                                         float* __restrict__ s) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float4 m = t[i];
        float l0, l1;
        eig2_vals(m.x, m.y, m.w, l0, l1);
        const float a0 = fabsf(l0), a1 = fabsf(l1);
        s[i] = fmaxf(a0, a1) - fminf(a0, a1);
    }
}

// Order-preserving float <-> unsigned key (for atomicMax on any finite float).
__device__ __forceinline__ unsigned fkey(float f) {
    const unsigned b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float fkey_inv(unsigned k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

__global__ __launch_bounds__(256) void k_otsu_max(const float* __restrict__ v, size_t n, int stride,
                                                  unsigned* __restrict__ key) {
    __shared__ unsigned s_max[4];
    unsigned m = 0;
    const size_t step = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {  // four reads in flight
        const float a = v[i * stride], b = v[(i + step) * stride], c = v[(i + 2 * step) * stride],
                    d = v[(i + 3 * step) * stride];
        m = max(max(m, fkey(a)), max(fkey(b), max(fkey(c), fkey(d))));
    }
    for (; i < n; i += step) m = max(m, fkey(v[i * stride]));
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
    __syncthreads();
    // one atomic per block: one per wave of 4096 blocks took 198 us over 12.6 M values
    if (threadIdx.x == 0) atomicMax(key, max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3])));
}

// numpy.histogram(values, 256, range=(0, vmax)) for float32 values: float32
// edges = float32(i * vmax / 256), index from the float64 quotient, then the
// +-1 corrections at the edges; the last bin is closed.
__global__ __launch_bounds__(256) void k_otsu_hist(const float* __restrict__ v, size_t n, int stride,
                                                   const unsigned* __restrict__ key,
                                                   unsigned long long* __restrict__ hist) {
    // a histogram per wave: most values of a saliency fall into the first bins
    __shared__ unsigned hw[4][256];
    __shared__ float edge[257];
    const float vmax = fkey_inv(*key);
    const double dv = (double)vmax, step = dv / 256.0;
#pragma unroll
    for (int k = 0; k < 4; k++) hw[k][threadIdx.x] = 0;
    edge[threadIdx.x] = (float)((double)threadIdx.x * step);
    if (threadIdx.x == 0) edge[256] = vmax;
    __syncthreads();
    unsigned* h = hw[threadIdx.x >> 6];
    // The quotient's bin and its corrections by one amount to the bin whose
    // edges enclose the value: found from an FP32 quotient and the edges where
    // those are distinct floats, else by the FP64 steps themselves. VALU-bound:
    // 58 us over 12.6 M values (61 us with FP64 quotients and an LDS atomic per
    // value), where reading them takes 25.
    const bool distinct = vmax > 1e-30f;
    const float inv = distinct ? 256.0f / vmax : 0.0f;
    auto bin = [&](float a) {  // -1: outside the range
        if (!(a >= 0.0f && a <= vmax)) return -1;
        int idx;
        if (distinct) {
            idx = min((int)(a * inv), 255);
            while (a < edge[idx]) idx--;  // edge[0] = 0 <= a
            while (idx != 255 && a >= edge[idx + 1]) idx++;
        } else {
            idx = (int)(((double)a / dv) * 256.0);
            if (idx == 256) idx = 255;
            if (a < edge[idx]) idx--;
            if (idx != 255 && a >= edge[idx + 1]) idx++;
        }
        return idx;
    };
    // lanes that share a bin add once: equal LDS addresses would queue up
    auto add = [&](int idx) {
        for (int round = 0; round < 4; round++) {
            if (idx < 0) return;
            const int lead = __builtin_amdgcn_readfirstlane(idx);
            const unsigned long long same = __ballot(idx == lead);
            if (idx == lead) {
                if ((threadIdx.x & 63) == (unsigned)__builtin_ctzll(same)) atomicAdd(&h[lead], (unsigned)__popcll(same));
                return;
            }
        }
        atomicAdd(&h[idx], 1u);
    };
    if (vmax > 0.0f) {
        const size_t hop = (size_t)gridDim.x * blockDim.x;
        size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
        for (; i + 3 * hop < n; i += 4 * hop) {  // four reads in flight
            const float a0 = v[i * stride], a1 = v[(i + hop) * stride], a2 = v[(i + 2 * hop) * stride],
                        a3 = v[(i + 3 * hop) * stride];
            add(bin(a0));
            add(bin(a1));
            add(bin(a2));
            add(bin(a3));
        }
        for (; i < n; i += hop) add(bin(v[i * stride]));
    }
    __syncthreads();
    const unsigned long long c = (unsigned long long)hw[0][threadIdx.x] + hw[1][threadIdx.x] + hw[2][threadIdx.x] +
                                 hw[3][threadIdx.x];
    if (c) atomicAdd(&hist[threadIdx.x], c);
}

// Otsu's between-class variance over the 256 bins, FP64, first maximum
// (reconstruct.py:46-63); threshold = that bin's float32 centre. The sums run
// in bin order (one thread, from LDS), the variances one per thread. One
// thread for all of it, each bin read from memory in turn, took 58 us.
__global__ __launch_bounds__(256) void k_otsu_select(const unsigned* __restrict__ key,
                                                     const unsigned long long* __restrict__ hist,
                                                     float* __restrict__ thr) {
    __shared__ double s_w[256], s_c[256], s_b[256];
    __shared__ float s_ctr[256];
    const int i = (int)threadIdx.x;
    const float vmax = fkey_inv(*key);
    if (!(vmax > 0.0f)) {
        if (i == 0) *thr = 0.0f;
        return;
    }
    const double step = (double)vmax / 256.0;
    const float e0 = (float)((double)i * step), e1 = i == 255 ? vmax : (float)((double)(i + 1) * step);
    s_ctr[i] = (e0 + e1) / 2.0f;
    s_w[i] = (double)hist[i];
    s_c[i] = s_w[i] * (double)s_ctr[i];
    __syncthreads();
    if (i == 0) {  // running sums in place: s_w[255] the total, s_c[255] mu_total
        double w = 0.0, c = 0.0;
        for (int k = 0; k < 256; k++) {
            w += s_w[k];
            c += s_c[k];
            s_w[k] = w;
            s_c[k] = c;
        }
    }
    __syncthreads();
    const double total = s_w[255], mu_total = s_c[255];
    if (total == 0.0) {
        if (i == 0) *thr = 0.0f;
        return;
    }
    {
        const double w0 = s_w[i], cum = s_c[i], w1 = total - w0;
        const double mu0 = w0 > 0 ? cum / w0 : 0.0;
        const double mu1 = w1 > 0 ? (mu_total - cum) / w1 : 0.0;
        const double d = mu0 - mu1;
        s_b[i] = w0 * w1 * (d * d);
    }
    __syncthreads();
    if (i == 0) {
        double best = s_b[0];
        int at = 0;
        for (int k = 1; k < 256; k++)
            if (s_b[k] > best) { best = s_b[k]; at = k; }
        *thr = s_ctr[at];
    }
}

__global__ __launch_bounds__(256) void k_threshold(const float* __restrict__ v, size_t n, int stride,
                                                   const float* __restrict__ thr, unsigned char* __restrict__ mask) {
    const float t = *thr;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        mask[i] = v[i * stride] > t ? 1 : 0;
}

static unsigned grid_for(size_t n, unsigned per_block = 256, unsigned cap = 8192) {
    return (unsigned)std::max<size_t>(1, std::min<size_t>(ceil_div(n, per_block), cap));
}

// ---------------------------------------------------------------- host drivers
int otsu_run(const float* v, size_t n, int stride, float* thr, hipStream_t st) {
    unsigned* key = nullptr;
    TH_TRY(ws_get(WS_COUNTER, 8 + 256 * 8 + 64, (void**)&key));
    unsigned long long* hist = (unsigned long long*)((char*)key + 64);
    k_fill_u64<<<1, 256, 0, st>>>(hist, 256);
    k_thin_zero<<<1, 64, 0, st>>>(key, 1);
    ProfScope prof("otsu", st);
    k_otsu_max<<<grid_for(n, 256 * 16, 1024), 256, 0, st>>>(v, n, stride, key);
    k_otsu_hist<<<grid_for(n, 256 * 16, 512), 256, 0, st>>>(v, n, stride, key, hist);
    k_otsu_select<<<1, 256, 0, st>>>(key, hist, thr);
    TH_HIP(hipGetLastError());
    return TIRA_OK;
}

constexpr int kThinSlots = 4;   // per direction: its candidates, whether each re-check launch changed a mark
constexpr int kThinRounds = 4;  // re-evaluations per re-check launch but the verifying one

// Lee thinning of the 0/1 byte volume `v` (device) in place; blocking. The
// object voxels are compacted into a list once and the list is refiltered
// after every outer pass, so each border direction examines the remaining
// object voxels only instead of the whole volume.
//
// An outer pass is queued whole: per direction the candidates, two re-checks of
// kThinRounds rounds, one that verifies them, and the deletions, then the next
// object list, and the host reads the pass's counters once. A direction whose
// re-check had not settled applies nothing and makes the rest of the pass do
// nothing; the host then repeats its re-check until it settles and queues the
// directions after it. A read-back after every direction and Jacobi sweeps of
// one evaluation a launch took 2.2 ms where this takes 1.0 (192 x 256 x 256
// vessels, 5 outer passes); with one re-check and its verification a direction
// in eight was taken up again.
int lee_run(unsigned char* v, unsigned s0, unsigned s1, unsigned s2, unsigned* iterations, hipStream_t st) {
    const size_t n = (size_t)s0 * s1 * s2;
    unsigned char* mark = nullptr;
    unsigned *list = nullptr, *cnt = nullptr, *objA = nullptr, *objB = nullptr;
    // [0 .. 5] whether a direction deleted a voxel, [6] object voxels, [7] stall, then per
    // direction kThinSlots
    constexpr int kObj = 6, kStall = 7, kDir = 8, kAll = kDir + 6 * kThinSlots;
    TH_TRY(ws_get(WS_SCRATCH0, n, (void**)&mark));
    TH_TRY(ws_get(WS_COUNTER, kAll * 4, (void**)&cnt));
    k_fill_u8<<<grid_for(n), 256, 0, st>>>(mark, n);
    TH_HIP(hipGetLastError());
    ProfScope prof("lee_thin", st);
    // object list: count, size the buffers, gather
    const bool aligned = ((uintptr_t)v & 15) == 0;
    const size_t per = std::max<size_t>((n / 1024 + 4095) & ~size_t(4095), 4096);
    auto objects = [&](unsigned* to) -> int {
        k_thin_zero<<<1, 64, 0, st>>>(cnt + kObj, 2);
        if (aligned) k_thin_objects_vol<<<(unsigned)((n + per - 1) / per), 256, 0, st>>>(v, n, per, to, cnt + kObj);
        else k_thin_objects<<<grid_for(n), 256, 0, st>>>(v, nullptr, n, to, cnt + kObj, nullptr);
        TH_HIP(hipGetLastError());
        return TIRA_OK;
    };
    unsigned host[8];
    TH_TRY(objects(nullptr));
    TH_HIP(hipMemcpyAsync(host + kObj, cnt + kObj, 4, hipMemcpyDeviceToHost, st));
    TH_HIP(hipStreamSynchronize(st));
    unsigned nobj = host[kObj];
    if (nobj == 0) {
        if (iterations) *iterations = 1;  // one outer pass finds nothing to delete
        return TIRA_OK;
    }
    TH_TRY(ws_get(WS_SCRATCH2, (size_t)nobj * 4, (void**)&list));
    TH_TRY(ws_get(WS_THIN0, (size_t)nobj * 4, (void**)&objA));
    TH_TRY(ws_get(WS_THIN1, (size_t)nobj * 4, (void**)&objB));
    TH_TRY(objects(objA));
    // The candidates' neighbourhood codes go to objB, which is free until the
    // pass's object list is rebuilt. The re-check and apply passes read the
    // candidate count on the device (launched over the object count, an upper
    // bound).
    auto resolve = [&](unsigned* dc, unsigned* ch, const unsigned* prev, int rounds) {
        k_thin_resolve<<<grid_for(nobj), 256, 0, st>>>((int)s1, (int)s2, list, objB, dc, mark, ch, prev, rounds);
    };
    int iters = 0;
    for (;;) {
        iters++;
        k_thin_zero_n<<<1, 256, 0, st>>>(cnt, kAll);
        for (int first = 0; first < 6;) {
            for (int dir = first; dir < 6; dir++) {
                unsigned* dc = cnt + kDir + dir * kThinSlots;
                k_thin_candidates_list<<<grid_for(nobj), 256, 0, st>>>(v, (int)s0, (int)s1, (int)s2, dir, objA, nobj,
                                                                       mark, list, objB, dc, cnt + kStall);
                resolve(dc, dc + 1, nullptr, kThinRounds);
                resolve(dc, dc + 2, dc + 1, kThinRounds);
                resolve(dc, dc + 3, dc + 2, 1);
                k_thin_apply<<<grid_for(nobj), 256, 0, st>>>(v, list, dc, mark, cnt + dir, dc + 3, cnt + kStall,
                                                             (unsigned)dir + 1);
                TH_HIP(hipGetLastError());
            }
            // drop deleted voxels from the object list; read it with this pass's deletions
            k_thin_objects<<<grid_for(nobj), 256, 0, st>>>(v, objA, nobj, objB, cnt + kObj, cnt + kStall);
            TH_HIP(hipGetLastError());
            TH_HIP(hipMemcpyAsync(host, cnt, 8 * 4, hipMemcpyDeviceToHost, st));
            TH_HIP(hipStreamSynchronize(st));
            if (!host[kStall]) break;
            const int dir = (int)host[kStall] - 1;
            unsigned* dc = cnt + kDir + dir * kThinSlots;
            // bounded: each launch settles at least one more level of the raster-order DAG, and
            // there are at most nobj candidates
            for (unsigned k = 0;; k++) {
                TH_ARG(k <= nobj, "thinning re-check did not settle (internal error)");
                k_thin_zero<<<1, 64, 0, st>>>(dc + 1, 2);
                resolve(dc, dc + 1, nullptr, kThinRounds);
                resolve(dc, dc + 2, dc + 1, 1);
                TH_HIP(hipGetLastError());
                TH_HIP(hipMemcpyAsync(host, dc + 2, 4, hipMemcpyDeviceToHost, st));
                TH_HIP(hipStreamSynchronize(st));
                if (host[0] == 0) break;
            }
            k_thin_apply<<<grid_for(nobj), 256, 0, st>>>(v, list, dc, mark, cnt + dir, nullptr, nullptr, 0u);
            k_thin_zero<<<1, 64, 0, st>>>(cnt + kObj, 2);
            TH_HIP(hipGetLastError());
            first = dir + 1;
            if (first == 6) {  // only the object list is left
                k_thin_objects<<<grid_for(nobj), 256, 0, st>>>(v, objA, nobj, objB, cnt + kObj, nullptr);
                TH_HIP(hipGetLastError());
                TH_HIP(hipMemcpyAsync(host, cnt, 8 * 4, hipMemcpyDeviceToHost, st));
                TH_HIP(hipStreamSynchronize(st));
            }
        }
        bool deleted_any = false;
        for (int d = 0; d < 6; d++) deleted_any = deleted_any || host[d] != 0;
        if (!deleted_any) break;  // a whole pass of six directions deleted nothing
        nobj = host[kObj];
        std::swap(objA, objB);
        if (nobj == 0) {  // the next outer pass would find no candidate in any direction
            iters++;
            break;
        }
    }
    if (iterations) *iterations = (unsigned)iters;
    return TIRA_OK;
}

}  // namespace th

using namespace th;

extern "C" {

int tira_stick_saliency2_async(const float* field4, size_t n, float* saliency) {
    TH_ARG(field4 && saliency, "NULL pointer");
    if (!n) return TIRA_OK;
    hipStream_t st = stream();
    k_stick_saliency2<<<grid_for(n), 256, 0, st>>>((const float4*)field4, n, saliency);
    TH_HIP(hipGetLastError());
    return TIRA_OK;
}

int tira_otsu_threshold_async(const float* values, size_t n, int stride, float* threshold) {
    TH_ARG(values && threshold, "NULL pointer");
    TH_ARG(stride >= 1, "stride must be >= 1");
    TH_ARG(n >= 1, "Otsu needs at least one value");
    return otsu_run(values, n, stride, threshold, stream());
}

int tira_threshold_async(const float* values, size_t n, int stride, const float* threshold, unsigned char* mask) {
    TH_ARG(values && threshold && mask, "NULL pointer");
    TH_ARG(stride >= 1, "stride must be >= 1");
    if (!n) return TIRA_OK;
    hipStream_t st = stream();
    k_threshold<<<grid_for(n), 256, 0, st>>>(values, n, stride, threshold, mask);
    TH_HIP(hipGetLastError());
    return TIRA_OK;
}

int tira_lee_thin3_u8(unsigned char* mask, unsigned s0, unsigned s1, unsigned s2, unsigned* iterations) {
    TH_ARG(mask, "NULL pointer");
    TH_ARG((size_t)s0 * s1 * s2 < ((size_t)1 << 32), "volume too large for 32-bit voxel indices");
    TH_ARG(is_device(mask), "tira_lee_thin3_u8 takes a device pointer");
    const size_t n = (size_t)s0 * s1 * s2;
    if (!n) { if (iterations) *iterations = 0; return TIRA_OK; }
    hipStream_t st = stream();
    k_thin_binarise<unsigned char><<<grid_for(n), 256, 0, st>>>(mask, mask, n);
    TH_HIP(hipGetLastError());
    return lee_run(mask, s0, s1, s2, iterations, st);
}

int tira_lee_thin3(const int* in, int* out, unsigned x, unsigned y, unsigned z, unsigned* iterations) {
    TH_ARG(in && out, "NULL pointer");
    const size_t n = (size_t)x * y * z;
    TH_ARG(n < ((size_t)1 << 32), "volume too large for 32-bit voxel indices");
    if (!n) { if (iterations) *iterations = 0; return TIRA_OK; }
    const int* din; void* dout;
    TH_TRY(stage_in(in, n * 4, WS_IN0, (const void**)&din));
    TH_TRY(stage_out(out, n * 4, WS_OUT0, &dout));
    unsigned char* v = nullptr;
    TH_TRY(ws_get(WS_PIPE0, n, (void**)&v));
    hipStream_t st = stream();
    k_thin_binarise<int><<<grid_for(n), 256, 0, st>>>(din, v, n);
    TH_HIP(hipGetLastError());
    TH_TRY(lee_run(v, z, y, x, iterations, st));
    k_thin_export<int><<<grid_for(n), 256, 0, st>>>(v, (int*)dout, n);
    TH_HIP(hipGetLastError());
    return finish_out(out, dout, n * 4);
}

int tira_thin3_classify_async(unsigned first, unsigned count, unsigned char* flags) {
    TH_ARG(flags, "NULL pointer");
    TH_ARG((unsigned long long)first + count <= (1ull << 26), "codes beyond 2^26");
    if (!count) return TIRA_OK;
    hipStream_t st = stream();
    k_thin_classify<<<grid_for(count), 256, 0, st>>>(first, count, flags);
    TH_HIP(hipGetLastError());
    return TIRA_OK;
}

// Voted field -> magnitude-ranked saliency (eig3) -> Otsu threshold of the
// stick saliency -> mask -> Lee thinning. Device pointers; blocking (the
// thinning loop reads counters back).
int tira_skeleton3(const float* voted, int layout, unsigned s0, unsigned s1, unsigned s2, float* saliency3,
                   float* threshold, unsigned char* skeleton, unsigned* iterations) {
    TH_ARG(voted && saliency3 && threshold && skeleton, "NULL pointer");
    TH_ARG(layout == TIRA_LAYOUT_MAT9 || layout == TIRA_LAYOUT_PACKED6, "bad layout");
    TH_ARG(is_device(voted) && is_device(saliency3) && is_device(threshold) && is_device(skeleton),
           "tira_skeleton3 takes device pointers");
    const size_t n = (size_t)s0 * s1 * s2;
    TH_ARG(n >= 1, "empty volume");
    TH_ARG(n < ((size_t)1 << 32), "volume too large for 32-bit voxel indices");
    TH_TRY(tira_eig3_async(voted, n, layout, saliency3, nullptr, nullptr,
                           TIRA_EIG_SALIENCY | TIRA_EIG_MAGNITUDE | TIRA_EIG_REFINE_FP64 | TIRA_EIG_SCALE_INVARIANT,
                           nullptr));
    hipStream_t st = stream();
    TH_TRY(otsu_run(saliency3, n, 3, threshold, st));
    k_threshold<<<grid_for(n), 256, 0, st>>>(saliency3, n, 3, threshold, skeleton);
    TH_HIP(hipGetLastError());
    return lee_run(skeleton, s0, s1, s2, iterations, st);
}

}  // extern "C"
