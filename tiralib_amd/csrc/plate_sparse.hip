// plate_sparse.hip -- the tabulated learned-plate vote over the voters that
// carry a plate, instead of over every offset of every receiver's window.
//
// A voter of zero plate scale adds exactly nothing, and in the fields this
// vote serves most voxels are such (curved sheets with 2% plate noise: 4% of
// 256^3 voxels vote). The window gather (k_vote3_mlptab) evaluates all w^3
// pairs of a receiver; this one lists the voting voxels once and evaluates
// only pairs with a listed voter. Per field, tile by tile, the cheaper of the
// two is taken on the device (k_plate_tiles), so a dense field runs as before.
//
// List: the voters of every 64-voxel x segment in x order, segments in the
// order (x block, z, y), so the voters of a box are one contiguous run per
// (x block, z). A wave owns a 4 x 4 x 4 cube of receivers (one per lane): it
// loads 64 list entries at a time, keeps those inside the cube's box with a
// ballot and walks the set bits; a voter's values are broadcast from the lane
// that loaded them, so the voter is wave-uniform and the offset varies by
// lane. The offset's direction, attenuation and distance row come from a
// table indexed by the offset (padded by the cube's edge: entries outside the
// window have row -1 and their lanes sit the pair out), the network's rows
// from LDS.
#include "common.hpp"
#include "plate_sparse.hpp"
#include "seg_list.hpp"
#include "vote3_acc.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace th {

constexpr int kCube = 4;                     // receivers per cube edge, 4^3 = one wave
constexpr int kSparseThreads = 1024;         // one block per CU (its LDS holds the table)
constexpr int kSparseCells = kMlpTabM + 2;   // staged cells of a row: x_j, j = -1 .. kMlpTabM
constexpr size_t kSparseLds = 160 * 1024 - 1024;

unsigned plate_sparse_max_rows() { return (unsigned)(kSparseLds / (kSparseCells * sizeof(float4))); }

// Voters of each segment: one wave per segment.
__global__ __launch_bounds__(256) void k_plate_count(const float4* __restrict__ pay, VoteGeom g, unsigned nseg,
                                                     unsigned* __restrict__ cnt) {
    const unsigned seg = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (seg > nseg) return;
    if (seg == nseg) {  // the end of the list
        if (lane == 0) cnt[seg] = 0;
        return;
    }
    const unsigned y = seg % (unsigned)g.s1, zx = seg / (unsigned)g.s1;
    const unsigned z = zx % (unsigned)g.s0, x = zx / (unsigned)g.s0 * 64 + lane;
    bool on = false;
    if (x < (unsigned)g.s2) on = pay[((size_t)(z + g.r) * g.P1 + y + g.r) * g.P2 + x + g.r].w != 0.0f;
    const unsigned long long m = __ballot(on);
    if (lane == 0) cnt[seg] = (unsigned)__popcll(m);
}

// The list: voter (n, scale) and position (x + (y << 16), z).
__global__ __launch_bounds__(256) void k_plate_list(const float4* __restrict__ pay, VoteGeom g, unsigned nseg,
                                                    const unsigned* __restrict__ cnt, const unsigned* __restrict__ tot,
                                                    float4* __restrict__ lv, uint2* __restrict__ lp) {
    const unsigned seg = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (seg >= nseg) return;
    const unsigned y = seg % (unsigned)g.s1, zx = seg / (unsigned)g.s1;
    const unsigned z = zx % (unsigned)g.s0, x = zx / (unsigned)g.s0 * 64 + lane;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (x < (unsigned)g.s2) v = pay[((size_t)(z + g.r) * g.P1 + y + g.r) * g.P2 + x + g.r];
    const unsigned long long m = __ballot(v.w != 0.0f);
    if (v.w != 0.0f) {
        const unsigned k = seg_start(cnt, tot, seg) + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
        lv[k] = v;
        lp[k] = make_uint2(x | (y << 16), z);
    }
}

// Per receiver tile of the window gather (64 x 4 x bz): 1 when its voters are
// few enough that the listed gather is the cheaper. One wave per tile. The
// listed gather evaluates every listed voter of a cube's box on 64 lanes
// ((2r + 4)^3 offsets for the w^3 of the window), the window gather all w^3
// offsets of the 64 lanes: `ratio` is the cost of a listed pair over that of
// a window pair.
__global__ __launch_bounds__(256) void k_plate_tiles(VoteGeom g, int bz, const unsigned* __restrict__ cnt,
                                                     const unsigned* __restrict__ tot, float ratio,
                                                     unsigned char* __restrict__ sparse, unsigned* __restrict__ dense) {
    const unsigned t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const unsigned nt = g.nbx * g.nby * g.nbz;
    if (t >= nt) return;
    const int x0 = (int)(t % g.nbx) * 64, y0 = (int)((t / g.nbx) % g.nby) * 4, z0 = (int)(t / (g.nbx * g.nby)) * bz;
    const int ylo = max(y0 - g.r, 0), yhi = min(y0 + 4 + g.r, g.s1);
    const int zlo = max(z0 - g.r, 0), zhi = min(z0 + bz + g.r, g.s0);
    const int xlo = max(x0 - g.r, 0) / 64, xhi = min(x0 + 63 + g.r, g.s2 - 1) / 64;
    unsigned c = 0;
    for (int z = zlo + (int)lane; z < zhi; z += 64)
        for (int xb = xlo; xb <= xhi; xb++) {
            const unsigned row = ((unsigned)xb * g.s0 + z) * g.s1;
            c += seg_start(cnt, tot, row + yhi) - seg_start(cnt, tot, row + ylo);
        }
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d);
    if (lane == 0) {
        const float box = (float)(xhi - xlo + 1) * 64.0f * (float)(4 + 2 * g.r) * (float)(bz + 2 * g.r);
        const float wc = (float)(2 * g.r + kCube), ww = (float)(2 * g.r + 1);
        const bool few = (float)c * wc * wc * wc * ratio < box * ww * ww * ww;
        sparse[t] = few ? 1 : 0;
        if (dense && !few) atomicAdd(dense, 1u);
    }
}

// One offset's entry: unit direction d and c1 / pi, and the byte offset of
// its row in LDS, negative outside the window.
struct Entry {
    float4 d;
    int row;
};
// Entry `sbase + lane_off` (sbase wave-uniform: it goes into the scalar base
// address, so the loads take no vector address arithmetic).
__device__ __forceinline__ void fetch(const float4* __restrict__ ent, const int* __restrict__ entrow, int sbase,
                                      unsigned lane_off, Entry& e) {
    const char* pe = (const char*)(ent + (unsigned)sbase);
    const char* pr = (const char*)(entrow + (unsigned)sbase);
    e.d = *(const float4*)(pe + lane_off * 16u);
    e.row = *(const int*)(pr + lane_off * 4u);
}

// w c [A I + B n n^T + G (n d^T + d n^T) + 2 H d d^T] of voter (n, w) at entry
// e, with h = G n + H d: h d^T + d h^T, whose diagonal goes to hd at half its value.
__device__ __forceinline__ void listed_pair(Acc& a, float3& hd, float nx, float ny, float nz, float w, const Entry& e,
                                            const float4* s_tab) {
    if (e.row < 0) return;
    const float dx = e.d.x, dy = e.d.y, dz = e.d.z;
    const float s = fmaf(nx, dx, fmaf(ny, dy, nz * dz));
    const float x = fmaf(-s, s, 1.0f);
    const float t = fmaf(x, (float)kMlpTabM, 0.5f);
    const float4* c = (const float4*)((const char*)s_tab + (((int)t << 4) + e.row));
    const float f = __builtin_amdgcn_fractf(t);
    const float4 c0 = c[0], c1 = c[1];
    const float A = fmaf(f, c1.x - c0.x, c0.x), B = fmaf(f, c1.y - c0.y, c0.y);
    const float G = s * fmaf(f, c1.z - c0.z, c0.z), H = fmaf(f, c1.w - c0.w, c0.w);
    const float wc = w * e.d.w;
    const float n0 = wc * nx, n1 = wc * ny, n2 = wc * nz;
    a.ii = fmaf(wc, A, a.ii);
    const float b0 = B * n0, b1 = B * n1, b2 = B * n2;
    a.xx = fmaf(b0, nx, a.xx); a.xy = fmaf(b0, ny, a.xy); a.xz = fmaf(b0, nz, a.xz);
    a.yy = fmaf(b1, ny, a.yy); a.yz = fmaf(b1, nz, a.yz); a.zz = fmaf(b2, nz, a.zz);
    const float Hw = wc * H;
    const float h0 = fmaf(Hw, dx, G * n0), h1 = fmaf(Hw, dy, G * n1), h2 = fmaf(Hw, dz, G * n2);
    hd.x = fmaf(h0, dx, hd.x); hd.y = fmaf(h1, dy, hd.y); hd.z = fmaf(h2, dz, hd.z);
    a.xy = fmaf(h0, dy, fmaf(h1, dx, a.xy));
    a.xz = fmaf(h0, dz, fmaf(h2, dx, a.xz));
    a.yz = fmaf(h1, dz, fmaf(h2, dy, a.yz));
}

// The listed gather. Persistent blocks, one per CU: 130 KB of LDS hold the
// rows of the network table (values at x_j; a lookup interpolates between two
// neighbouring cells), every wave takes cubes from a counter until none is
// left. VALU-bound: 58 instructions per (cube, voter), 84% of the issue slots
// in use, 71% of the lanes inside the window at w = 25 (a 4 x 4 x 8 box on two
// receivers per lane would have 62%). 256^3 curved sheets with 2% plate noise,
// w = 25: 27 ms (30 ms with the entry addresses in vector arithmetic and the
// prefetched entry copied), where the window gather of stick and plate took
// 285 ms; the sticks take 5.9 ms as a spectral vote in FP64.
__global__ __launch_bounds__(kSparseThreads) void k_plate_sparse(
    const float4* __restrict__ lv, const uint2* __restrict__ lp, const unsigned* __restrict__ cnt,
    const unsigned* __restrict__ tot, const float4* __restrict__ ent, const int* __restrict__ entrow,
    const float4* __restrict__ vtab, const int* __restrict__ rows, int nrows, VoteGeom g, int bz,
    const unsigned char* __restrict__ sparse, unsigned* __restrict__ next, float* __restrict__ out, int layout,
    int accumulate, const unsigned long long* __restrict__ stop) {
    if (stop && *stop) return;
    extern __shared__ float4 s_tab[];
    for (int i = (int)threadIdx.x; i < nrows * kSparseCells; i += kSparseThreads) {
        const int slot = i / kSparseCells, p = i - slot * kSparseCells;
        // cell p holds x_(p-1); the end segments continue linearly
        const int o = min(max(p - 1, 0), kMlpTabM - 2);
        const float4* src = vtab + ((size_t)rows[slot] * kMlpTabM + o) * 2;
        const float4 v = src[0], dl = src[1];
        const float sh = (float)(p - 1 - o);
        s_tab[i] = make_float4(fmaf(sh, dl.x, v.x), fmaf(sh, dl.y, v.y), fmaf(sh, dl.z, v.z), fmaf(sh, dl.w, v.w));
    }
    __syncthreads();
    const int lane = (int)threadIdx.x & 63;
    const int xl = lane & 3, yl = (lane >> 2) & 3, zl = lane >> 4;
    const int r = g.r, D = 2 * r + 2 * kCube - 1;
    const unsigned lane_off = (unsigned)(((kCube - 1 - zl) * D + (kCube - 1 - yl)) * D + (kCube - 1 - xl));
    const unsigned ncx = ((unsigned)g.s2 + kCube - 1) / kCube, ncy = ((unsigned)g.s1 + kCube - 1) / kCube,
                   ncz = ((unsigned)g.s0 + kCube - 1) / kCube, ncube = ncx * ncy * ncz;
    for (;;) {
        unsigned item = 0;
        if (lane == 0) item = atomicAdd(next, 1u);
        item = (unsigned)__builtin_amdgcn_readfirstlane((int)item);
        if (item >= ncube) break;
        const int z0 = (int)(item % ncz) * kCube, x0 = (int)((item / ncz) % ncx) * kCube,
                  y0 = (int)(item / (ncz * ncx)) * kCube;
        if (!sparse[((unsigned)(z0 / bz) * g.nby + (unsigned)(y0 / 4)) * g.nbx + (unsigned)(x0 / 64)]) continue;
        const int ylo = max(y0 - r, 0), yhi = min(y0 + kCube + r, g.s1);
        const int zlo = max(z0 - r, 0), zhi = min(z0 + kCube + r, g.s0);
        const int xlo = max(x0 - r, 0), xhi = min(x0 + kCube - 1 + r, g.s2 - 1);
        Acc sum{0, 0, 0, 0, 0, 0, 0};
        for (int z = zlo; z < zhi; z++) {
            // a plane's votes are summed apart and added once: 2.3e-7 from the
            // 64-bit sum of the same table at 256^3, w = 25, where one running
            // sum over the box had 1.9e-6 and the window gather 1.4e-6
            Acc a{0, 0, 0, 0, 0, 0, 0};
            float3 hd = make_float3(0.0f, 0.0f, 0.0f);
            for (int xb = xlo / 64; xb <= xhi / 64; xb++) {
                const unsigned seg = ((unsigned)xb * g.s0 + z) * g.s1;
                const unsigned k0 = seg_start(cnt, tot, seg + ylo), k1 = seg_start(cnt, tot, seg + yhi);
                for (unsigned kb = k0; kb < k1; kb += 64) {
                    const unsigned k = kb + lane;
                    int vx = 0, vy = 0;
                    bool in = false;
                    if (k < k1) {
                        const uint2 q = lp[k];
                        vx = (int)(q.x & 0xffffu);
                        vy = (int)(q.x >> 16);
                        in = vx >= xlo && vx <= xhi;
                    }
                    unsigned long long m = __ballot(in);
                    if (!m) continue;
                    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    if (in) v = lv[k];
                    // offset-table index of the voter at the cube's far corner
                    const int base = ((z - z0 + r) * D + (vy - y0 + r)) * D + (vx - x0 + r);
                    // two entries in turn: the next voter's is in flight while
                    // this one is evaluated, and none is copied
                    Entry ea, eb;
                    int ja = __builtin_ctzll(m), jb = 0;
                    fetch(ent, entrow, __builtin_amdgcn_readlane(base, ja), lane_off, ea);
                    for (;;) {
                        m &= m - 1;
                        if (m) {
                            jb = __builtin_ctzll(m);
                            fetch(ent, entrow, __builtin_amdgcn_readlane(base, jb), lane_off, eb);
                        }
                        listed_pair(a, hd, lane_f(v.x, ja), lane_f(v.y, ja), lane_f(v.z, ja), lane_f(v.w, ja), ea, s_tab);
                        if (!m) break;
                        m &= m - 1;
                        if (m) {
                            ja = __builtin_ctzll(m);
                            fetch(ent, entrow, __builtin_amdgcn_readlane(base, ja), lane_off, ea);
                        }
                        listed_pair(a, hd, lane_f(v.x, jb), lane_f(v.y, jb), lane_f(v.z, jb), lane_f(v.w, jb), eb, s_tab);
                        if (!m) break;
                    }
                }
            }
            sum.xx += fmaf(2.0f, hd.x, a.xx); sum.yy += fmaf(2.0f, hd.y, a.yy); sum.zz += fmaf(2.0f, hd.z, a.zz);
            sum.xy += a.xy; sum.xz += a.xz; sum.yz += a.yz; sum.ii += a.ii;
        }
        const int x = x0 + xl, y = y0 + yl, z = z0 + zl;
        if (x < g.s2 && y < g.s1 && z < g.s0)
            write_out(out, layout, ((size_t)z * g.s1 + y) * g.s2 + x, sum, accumulate != 0);
    }
}

// ---------------------------------------------------------------- host
// Offset tables of the listed gather for (w, sigma1): direction and c1 / pi of
// every offset, its row's first LDS cell (-1 outside the window), and the
// network rows in use. Kept per host thread while the parameters and the
// buffer are unchanged.
struct SparseTabCache {
    int w = 0, nrows = 0;
    float s1 = 0.0f;
    int device = -1;
    void* ptr = nullptr;
    unsigned long long gen = 0;  // workspace generation: a released buffer may come back at its address
};
static thread_local SparseTabCache g_stab;

static int sparse_tables(int w, float s1, int vtab_rows, hipStream_t st, float4** ent, int** entrow, int** rows,
                         int* nrows) {
    const int r = w / 2, R = r + kCube - 1, D = 2 * R + 1;
    const size_t n = (size_t)D * D * D;
    const size_t bytes = n * 20 + (size_t)plate_sparse_max_rows() * 4;
    int dev = 0;
    TH_HIP(hipGetDevice(&dev));
    char* buf = nullptr;
    TH_TRY(ws_get(WS_TABLE5, bytes, (void**)&buf));
    *ent = (float4*)buf;
    *entrow = (int*)(buf + n * 16);
    *rows = (int*)(buf + n * 20);
    if (g_stab.w == w && g_stab.s1 == s1 && g_stab.device == dev && g_stab.ptr == buf &&
        g_stab.gen == ws_generation(WS_TABLE5)) {
        *nrows = g_stab.nrows;
        return TIRA_OK;
    }
    g_stab.device = -1;
    std::vector<int> shells, used, slot;
    mlp_shells(s1, shells);
    slot.assign(shells.size() + 2, -1);
    std::vector<char> h(bytes, 0);
    float4* he = (float4*)h.data();
    int* hr = (int*)(h.data() + n * 16);
    size_t k = 0;
    for (int dw = -R; dw <= R; dw++)
        for (int dv = -R; dv <= R; dv++)
            for (int du = -R; du <= R; du++, k++) {
                hr[k] = -1;
                if (std::abs(du) > r || std::abs(dv) > r || std::abs(dw) > r) continue;
                float d[3], c1, c2;
                offset_geometry(du, dv, dw, s1, 0.0f, d, c1, c2);
                he[k] = make_float4(d[0], d[1], d[2], (float)(c1 / M_PI));
                const int row = std::min(std::max(mlp_shell_row(shells, du * du + dv * dv + dw * dw), 0), vtab_rows - 1);
                if (slot[row] < 0) {
                    slot[row] = (int)used.size();
                    used.push_back(row);
                }
                hr[k] = slot[row] * kSparseCells * (int)sizeof(float4);
            }
    *nrows = (int)used.size();
    if (used.size() <= plate_sparse_max_rows()) std::copy(used.begin(), used.end(), (int*)(h.data() + n * 20));
    // ordered after earlier work on `st` that may still read the previous tables
    TH_HIP(hipStreamSynchronize(st));
    TH_HIP(hipMemcpy(buf, h.data(), bytes, hipMemcpyHostToDevice));
    g_stab.w = w; g_stab.s1 = s1; g_stab.nrows = *nrows; g_stab.device = dev; g_stab.ptr = buf;
    g_stab.gen = ws_generation(WS_TABLE5);
    return TIRA_OK;
}

// Cost of a listed (cube, voter) pair over a window pair of the plate part
// (see k_plate_tiles): 128^3 random plates, all voting, took 70.0 ms listed and
// 34.2 ms as windows at w = 25 (28^3 listed offsets for 25^3), 11.3 and 5.5 ms
// at w = 13 (16^3 for 13^3): 1.46 and 1.10. With 1.45 the listed form is taken
// up to a density of 0.49 at w = 25 (equal times measured at 0.46) and 0.37
// at w = 13 (0.47).
constexpr float kSparseRatio = 1.45f;

int plate_list_build(const float4* pay, int vtab_rows, float sigma1, const VoteGeom& g, int bz, unsigned* dense,
                     hipStream_t st, PlateList* list, bool* ok) {
    *ok = false;
    const size_t n = (size_t)g.s0 * g.s1 * g.s2;
    if (n >= (size_t)1 << 31 || g.s1 > 65535 || g.s2 > 65535) return TIRA_OK;
    const unsigned nseg = g.nbx * (unsigned)g.s0 * (unsigned)g.s1, ntile = g.nbx * g.nby * g.nbz;
    const unsigned nscan = (nseg + 1 + kScanSegs - 1) / kScanSegs;
    const size_t lv_b = n * 16, lp_b = n * 8, cnt_b = ((size_t)nseg + 1) * 4, tot_b = (size_t)nscan * 4;
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    char* buf = nullptr;
    PlateList& L = *list;
    int rc = sparse_tables(2 * g.r + 1, sigma1, vtab_rows, st, &L.ent, &L.entrow, &L.rows, &L.nrows);
    if (rc == TIRA_OK && L.nrows > (int)plate_sparse_max_rows()) return TIRA_OK;
    if (rc == TIRA_OK) rc = ws_get(WS_LIST, up(lv_b) + up(lp_b) + up(cnt_b) + up(tot_b) + 256 + ntile, (void**)&buf);
    if (rc == TIRA_ERR_OUT_OF_MEMORY) {  // the window gather needs neither
        (void)hipGetLastError();
        return TIRA_OK;
    }
    TH_TRY(rc);
    L.lv = (float4*)buf;
    L.lp = (uint2*)(buf + up(lv_b));
    L.cnt = (unsigned*)(buf + up(lv_b) + up(lp_b));
    L.tot = (unsigned*)((char*)L.cnt + up(cnt_b));
    L.next = (unsigned*)((char*)L.tot + up(tot_b));
    L.sparse = (unsigned char*)L.next + 256;
    ProfScope prof("plate_list", st);
    k_plate_count<<<nseg / 4 + 1, 256, 0, st>>>(pay, g, nseg, L.cnt);
    k_seg_scan<<<nscan, 256, 0, st>>>(L.cnt, nseg + 1, L.tot);
    k_seg_scan_top<<<1, 1024, 0, st>>>(L.tot, nscan, L.next);
    k_plate_list<<<ceil_div(nseg, 4), 256, 0, st>>>(pay, g, nseg, L.cnt, L.tot, L.lv, L.lp);
    k_plate_tiles<<<ceil_div(ntile, 4), 256, 0, st>>>(g, bz, L.cnt, L.tot, kSparseRatio, L.sparse, dense);
    TH_HIP(hipGetLastError());
    *ok = true;
    return TIRA_OK;
}

int plate_sparse_gather(const PlateList& L, const float4* vtab, const VoteGeom& g, int bz, float* out, int layout,
                        bool accumulate, const unsigned long long* stop, hipStream_t st) {
    ProfScope prof("plate_sparse", st);
    const size_t lds = (size_t)L.nrows * kSparseCells * sizeof(float4);
    TH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_plate_sparse), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)kSparseLds));
    k_plate_sparse<<<(unsigned)cu_count(), kSparseThreads, lds, st>>>(L.lv, L.lp, L.cnt, L.tot, L.ent, L.entrow, vtab,
                                                                      L.rows, L.nrows, g, bz, L.sparse, L.next, out,
                                                                      layout, accumulate ? 1 : 0, stop);
    TH_HIP(hipGetLastError());
    return TIRA_OK;
}

}  // namespace th
