// Time step of the moment-coefficient representation (kRepMom) with LDS
// exchange: one workgroup owns a TX x TY tile of the xy-plane and marches over
// a chunk of z-planes. Each plane's coefficients are read once, by the thread
// of their column (a halo of one node around the tile by the first four
// waves); the thread expands them to the Q post-collision populations and
// writes those that move in x or y into LDS at the place of the node they
// stream to. After one barrier a node reads its incoming populations of that
// plane: the ones with c_z < 0 complete the plane below, which then applies
// its boundary condition, collides and stores; the others wait in registers.
#pragma once
#include "kernels_impl.h"

namespace vlbm {

constexpr int kTileX = 64;      // one wave per tile row

// Populations that leave their column: LDS array of each.
template <int Q> struct Moving {
    static constexpr bool is(int i) { return kCX[i] != 0 || kCY[i] != 0; }
    static constexpr int slot(int i) {
        int n = 0;
        for (int k = 0; k < i; k++) n += is(k);
        return n;
    }
    static constexpr int count() { return slot(Q); }
};

// LDS arrays hold TY rows of 64 nodes. A row is followed by one pad column and
// an array by one pad row: values leaving the tile land in a pad (x = 64 in
// the column behind the row, x = -1 in the one behind the row before, y = TY
// and y = -1 in the rows between two arrays), so every lane writes without a
// bounds test and rows stay conflict-free. Two arrays sets (one barrier per
// plane) where two workgroups per CU fit 160 KB with them, else one set and
// two barriers: 75.1 KB float D3Q19, 56.4 KB float D3Q27 (both 64 x 8),
// 42.1 KB and 62.9 KB double (64 x 4). 256^3, us a step with the kernel that
// rebuilt pulled populations at their receiver and with this one: D3Q19 Bingham
// duct 397 300, circular duct 514 415 to 421, D3Q27 plates 461 304, double D3Q19
// plates 160 x 160 x 128 271 163.
template <typename T, int Q> struct TileShape {
    static constexpr int TY = sizeof(T) == 4 ? 8 : 4;
    static constexpr int NT = kTileX * TY;
    static constexpr int RS = kTileX + 1;
    static constexpr int AS = (TY + 1) * RS;
    static constexpr int SET = Moving<Q>::count() * AS;
    static constexpr int LEAD = RS + 1;                  // row y = -1 of the first array
    static constexpr int SETS = 2 * (LEAD + 2 * SET) * (int)sizeof(T) <= 160 * 1024 ? 2 : 1;
    static constexpr int WORDS = LEAD + SETS * SET;
    // waves per SIMD the register allocation must allow: two 512-thread
    // workgroups per CU, or 256-thread ones that LDS bounds to two or three
    static constexpr int MIN_WAVES = sizeof(T) == 4 ? 4 : 2;
};

// Post-collision populations for a boundary condition: operator() the node's
// own (offset 0) from its coefficients in registers, memory() any node's from
// the source lattice.
template <int Q, typename T>
struct ColumnPC {
    T* c;
    T* wall_a;       // wall weights of the column and the wall they are of (0: none yet)
    int* wall_of;
    GlobalPC<Q, T, T, kRepMom> far;
    __device__ __forceinline__ T operator()(int i, int, int, int) const { return recon<Q, T, T>(i, c, 1); }
    __device__ __forceinline__ T memory(int i, int dx, int dy, int dz) const { return far(i, dx, dy, dz); }
    static constexpr bool kCoefs = true, kFaces = true, kPlates = false;
    // wall weights: the same on every plane, so read when the wall changes
    __device__ __forceinline__ void walls(bool inside) const {
        const int w = inside ? 1 : 2;
        if (*wall_of == w) return;
        *wall_of = w;
#pragma unroll
        for (int b = 0; b < kIbbDirs; b++) wall_a[b] = far.wall(b, inside);
    }
    __device__ __forceinline__ T wall(int b, bool) const { return wall_a[b]; }
    // The coefficients may change here, as far as the compiler knows: it does
    // not lift the populations of a whole loop out of it into registers.
    __device__ __forceinline__ void fence() const {
#pragma unroll
        for (int k = 0; k < kCoef; k++) asm volatile("" : "+v"(c[k]));
    }
    __device__ __forceinline__ void own(T* out) const {
#pragma unroll
        for (int k = 0; k < kCoef; k++) out[k] = c[k];
    }
    // the coefficient layout is refused for the rheometer, the one reader of held values
    __device__ __forceinline__ T held(int) const { return (T)0; }
};

__device__ __forceinline__ int wrap_mod(int v, int n) {
    v %= n;
    return v < 0 ? v + n : v;
}

// Tiles of a step: n = ceil(nx/TX) * ceil(ny/TY) * ceil(nz/zc), x fastest. The
// divisors keep the decomposition of a tile number on the scalar unit, and with
// it the whole z loop.
struct TileGrid {
    FastDiv ntx, ntxy;
    int nty, zc, n;
};

inline TileGrid tile_grid(int nx, int ny, int nz, int ty, int zc) {
    const uint32_t ntx = (uint32_t)((nx + kTileX - 1) / kTileX), nty = (uint32_t)((ny + ty - 1) / ty);
    TileGrid g;
    g.ntx = make_fastdiv(ntx);
    g.ntxy = make_fastdiv(ntx * nty);
    g.nty = (int)nty;
    g.zc = zc;
    g.n = (int)(ntx * nty * (uint32_t)((nz + zc - 1) / zc));
    return g;
}

// One step over the lattice, coefficient planes src -> dst (p.src, p.dst).
// Grid: 8 ceil(n / 8) workgroups of TX*TY threads for the n tiles.
template <int Q, typename T, int RHEO, bool MASK, bool IBM>
__global__ __launch_bounds__((TileShape<T, Q>::NT), (TileShape<T, Q>::MIN_WAVES)) void k_step_tile(
    const Params<T> p, const TileGrid tg) {
    using SH = TileShape<T, Q>;
    using MV = Moving<Q>;
    constexpr int TX = kTileX, TY = SH::TY, RS = SH::RS, AS = SH::AS;
    static_assert(TY >= 4, "the first four waves read the halo");
    __shared__ T sm[SH::WORDS];
    __shared__ uint32_t region[27];
    // Workgroups go to the 8 XCDs in turn (blockIdx mod 8), each XCD with its
    // own L2. Block b takes tile (b mod 8) ceil(n / 8) + b / 8 of the n tiles,
    // so x- and y-neighbouring tiles run on one XCD at about the same time
    // and share the cache lines of their halos (a tile row's x halo alone
    // fetches 2 extra lines). The grid is 8 ceil(n / 8) blocks.
    const uint32_t b = blockIdx.x % 8u * (((uint32_t)tg.n + 7u) / 8u) + blockIdx.x / 8u;
    if (b >= (uint32_t)tg.n) return;
    const uint32_t bxy = fdiv(b, tg.ntx), bz = fdiv(b, tg.ntxy);
    const int x0 = (int)(b - bxy * tg.ntx.d) * TX, y0 = (int)(bxy - bz * (uint32_t)tg.nty) * TY, z0 = (int)bz * tg.zc;
    const int z1 = min(z0 + tg.zc, p.nz);
    const int lx = (int)threadIdx.x % TX;
    const int ly = __builtin_amdgcn_readfirstlane((int)threadIdx.x / TX);
    const uint32_t plane = (uint32_t)p.nx * (uint32_t)p.ny;
    const T* src = (const T*)p.src;

    // threads past a ragged edge read the wrapped node: its populations are
    // the halo of the last column or row
    const int x = x0 + lx, y = y0 + ly;
    const bool active = x < p.nx && y < p.ny;
    const uint32_t off = (uint32_t)wrap_mod(y, p.ny) * (uint32_t)p.nx + (uint32_t)wrap_mod(x, p.nx);
    // halo: the rows below (wave 0) and above the tile (wave 1), and the
    // columns left (wave 2) and right of it (wave 3) with the corners
    const int hr = ly == 0 ? -1 : (ly == 1 ? TY : lx - 1);            // row and column of the halo node
    const int hc = ly == 2 ? -1 : (ly == 3 ? TX : lx);
    const bool halo = ly < 2 || (ly < 4 && lx < TY + 2);
    uint32_t hoff = 0;
    if (halo) hoff = (uint32_t)wrap_mod(y0 + hr, p.ny) * (uint32_t)p.nx + (uint32_t)wrap_mod(x0 + hc, p.nx);

    auto load = [&](T* r, uint32_t node) {
        const T* q = src + node;
#pragma unroll
        for (int k = 0; k < kCoef; k++) r[k] = q[(int64_t)k * p.stride];
    };

    Node<T> nd;
    nd.x = x; nd.y = y;
    nd.xm = x == 0 ? p.nx - 1 : x - 1;
    nd.xp = x == p.nx - 1 ? 0 : x + 1;
    nd.ym = y == 0 ? p.ny - 1 : y - 1;
    nd.yp = y == p.ny - 1 ? 0 : y + 1;

    // Everything a plane needs from memory is loaded a plane ahead of its use:
    // a load the collision waits for would wait for the coefficients in flight
    // too (loads return in order). Node words of box maps come from LDS.
    T c[kCoef], h[kCoef], below[kCoef];
    T low[Q], up[Q];                           // gathered so far: of plane s - 1, and c_z > 0 of plane s
    uint32_t word = 0, word_next = 0;          // node words of planes s - 1 and s
    T om = 0, om_next = 0;                     // power law: omega of planes s - 1 and s
    Force<T> F = const_force(p), F_next = F;   // IBM: force on the nodes of planes s - 1 and s
    T wall_a[kIbbDirs];                        // node maps: interpolated bounce-back of the column
    int wall_of = 0;
    bool flag = false;                         // IBM: the node of plane s is in a flagged tile
#pragma unroll
    for (int k = 0; k < kCoef; k++) h[k] = below[k] = (T)0;
#pragma unroll
    for (int b = 0; b < kIbbDirs; b++) wall_a[b] = (T)0;
#pragma unroll
    for (int i = 0; i < Q; i++) low[i] = up[i] = (T)0;
    if (!MASK) {
        if (threadIdx.x < 27) region[threadIdx.x] = p.region_word[threadIdx.x];
        __syncthreads();
        word_next = region[box_region(x, y, 1, p.nx, p.ny, 3)];     // of a plane inside
    }
    {
        const uint32_t zo = (uint32_t)wrap_mod(z0 - 1, p.nz) * plane;
        load(c, zo + off);
        if (halo) load(h, zo + hoff);
        if (IBM && active) flag = p.tile_flag[tile_of(p, x, y, z0)] != 0;
    }
    int set = 0;
    for (int s = z0 - 1; s <= z1; s++) {
        T out[Q];
        expand<Q, T>(c, out);
        T* at = sm + SH::LEAD + set * SH::SET + ly * RS + lx;
#pragma unroll
        for (int i = 1; i < Q; i++)
            if (MV::is(i)) at[MV::slot(i) * AS + kCY[i] * RS + kCX[i]] = out[i];
        if (halo) {
            T e[Q];
            expand<Q, T>(h, e);
            T* to = sm + SH::LEAD + set * SH::SET + hr * RS + hc;
            if (ly == 0) {
#pragma unroll
                for (int i = 1; i < Q; i++)
                    if (kCY[i] > 0) to[MV::slot(i) * AS + kCY[i] * RS + kCX[i]] = e[i];
            } else if (ly == 1) {
#pragma unroll
                for (int i = 1; i < Q; i++)
                    if (kCY[i] < 0) to[MV::slot(i) * AS + kCY[i] * RS + kCX[i]] = e[i];
            } else {
                // from a corner only the population into the tile
                auto into = [&](int i) { return (kCY[i] <= 0 || hr < TY) && (kCY[i] >= 0 || hr >= 0); };
                if (ly == 2) {
#pragma unroll
                    for (int i = 1; i < Q; i++)
                        if (kCX[i] > 0 && into(i)) to[MV::slot(i) * AS + kCY[i] * RS + kCX[i]] = e[i];
                } else {
#pragma unroll
                    for (int i = 1; i < Q; i++)
                        if (kCX[i] < 0 && into(i)) to[MV::slot(i) * AS + kCY[i] * RS + kCX[i]] = e[i];
                }
            }
        }
        T own[kCoef];
#pragma unroll
        for (int k = 0; k < kCoef; k++) own[k] = c[k];
        {
            // in flight until the next plane; past the last one every lane
            // reads node 0 (one line), as a branch would make the loaded
            // registers wait for their copies
            const bool more = s < z1;
            const uint32_t zo = more ? (uint32_t)(s + 1 == p.nz ? 0 : s + 1) * plane : 0u;
            load(c, more ? zo + off : 0u);
            if (halo && more) load(h, zo + hoff);
            if (active && more && s >= z0) {
                const uint32_t idx = (uint32_t)s * plane + off;
                if (MASK) word_next = p.mask[idx];
                if (RHEO == 2) om_next = p.omega_state[idx];
                if (IBM) {
                    F_next = const_force(p);
                    if (flag) F_next = Force<T>{p.ibm_fx[idx], p.ibm_fy[idx], p.ibm_fz[idx]};
                    if (s + 1 < z1) flag = p.tile_flag[tile_of(p, x, y, s + 1)] != 0;
                }
            }
        }
        __syncthreads();
        const T* from = sm + SH::LEAD + set * SH::SET + ly * RS + lx;
#pragma unroll
        for (int i = 0; i < Q; i++)
            if (kCZ[i] < 0) low[i] = MV::is(i) ? from[MV::slot(i) * AS] : out[i];
        if (s > z0 && active) {
            const int z = s - 1;
            nd.z = z;
            nd.zm = z == 0 ? p.nz - 1 : z - 1;
            nd.zp = z == p.nz - 1 ? 0 : z + 1;
            nd.idx = (uint32_t)z * plane + off;
            if (!MASK && (z == 0 || z == p.nz - 1)) word = region[box_region(x, y, z, p.nx, p.ny, p.nz)];
            if (w_used(word)) {
                if (w_scheme(word) != kNull)
                    apply_bc<Q, T, MASK>(low, p, nd, word, ColumnPC<Q, T>{below, wall_a, &wall_of, {p, nd}});
                collide_store<Q, T, RHEO, kRepMom, kRepMom>(p, nd.idx, low, IBM ? F : const_force(p), om);
            }
        }
        word = word_next;
        om = om_next;
        if (IBM) F = F_next;
#pragma unroll
        for (int k = 0; k < kCoef; k++) below[k] = own[k];
#pragma unroll
        for (int i = 0; i < Q; i++) {
            if (kCZ[i] < 0) continue;
            const T v = MV::is(i) ? from[MV::slot(i) * AS] : out[i];
            if (kCZ[i] == 0) {
                low[i] = v;
            } else {
                low[i] = up[i];
                up[i] = v;
            }
        }
        if (SH::SETS == 1) __syncthreads();
        else set ^= 1;
    }
}

// z-chunk per workgroup: 32 planes, fewer until the lattice has enough
// workgroups to fill the device in whole rounds (two per CU: 2,048 are 4 rounds).
// The number comes from a kernel with another tile loop and was not swept with
// this one; a chunk reads two planes more than it completes.
inline int tile_zchunk(int nx, int ny, int nz, int ty) {
    const long tiles = (long)((nx + kTileX - 1) / kTileX) * ((ny + ty - 1) / ty);
    int zc = 32;
    while (zc > 4 && tiles * ((nz + zc - 1) / zc) < 2048) zc /= 2;
    return zc < nz ? zc : nz;
}

}  // namespace vlbm
