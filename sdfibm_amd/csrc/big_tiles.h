// big_tiles.h -- the tile pass for solids whose cell tile is too large for the
// LDS bit rows of k_classify (more than 63 cells along x or more than 1024
// vertex rows), e.g. the 40-80-cell CSG solids of a polydisperse cloud: one
// workgroup per solid would make such a tile the step's long pole, so these
// tiles are spread over the whole chip.
//
// Included by interact.hip, inside its kernel namespace, after the helpers it
// uses (divmod_small, block_exscan2, block_reduce, uf_find, code_none,
// cell_force).  The results are those of the
// reference's enumeration (src/cellenumerator.cpp:6-78) for these solids, as
// for every other solid: the cells with >= 1 strictly inside vertex, connected
// through faces to the seed (the nearest cell if it has an inside vertex, else
// the first such cell in index order), ALL_INSIDE when all 8 are inside.  The
// outputs go where k_classify puts them -- tile codes at the tile's offset, the
// candidate list (ALL_INSIDE cells ascending, then the cut cells ascending) in
// the list buffer at the same offset, the two counts -- so k_fields reads these
// tiles like any other.  The list holds tile-local linear indices here (the
// small tiles' packed (i, j, k) does not fit 80-cell tiles).
//
// All big solids of a step are processed together.  A tile's cell rows along x are
// cut into units of up to 64 cells, a thread each, and everything up to the
// candidate lists works on 64-bit masks of a unit: the component is labelled by
// union-find over the runs of active cells in the units (a label per run, in the
// list buffer at the run's first cell), not over cells.  (Labels per cell, with a
// thread per cell looking at its neighbours, took 0.95 ms for 50 CSG solids of
// 40-80 cells, 2.0e7 tile cells.)  Flat index spaces laid out by one scan kernel;
// no host round trip, so the step stays capturable.
//   k_big_layout    offsets of each big solid's vertex words, units, their blocks; totals
//   k_big_vertices  strict inside test per tile vertex (FP64) -> bit words, a vertex row's
//                   words aligned; spheres, ellipsoids, boxes, CSG on rectilinear meshes a
//                   word per thread by row intervals, otherwise a wave per word
//   k_big_units     per unit: its active (>= 1 inside vertex) and all-inside masks; a label
//                   per run; the lowest active cell
//   k_big_hook      unions of the runs that overlap along y, z and across unit ends
//   k_big_compress  labels -> roots
//   k_big_reach     per unit: the cells of the runs in the seed's component, their counts
//                   within the unit block; a second look at every overlap checks the unions
//                   converged (EF_LABEL otherwise)
//   k_big_scan      per solid, the unit blocks' counts scanned in order: list offsets, the
//                   solid's counts and candidate chunks
//   k_big_write     per unit (a wave): codes (NaN outside the component, +inf ALL_INSIDE; the
//                   cut cells' come from k_big_force) and its part of the candidate list
//   k_big_chunks    chunks of candidates (the chunk size is a run-time choice), their offsets
//   k_big_force     fractions, codes and forcing per chunk; FP64 partial sums
//   k_big_ft        partials summed in a fixed order, a wave per solid (x rho_f)
//                   -> force/torque
#pragma once

constexpr int kBigPer = 16;                  // big solids per thread of k_big_chunks
constexpr int kBigMaxSolids = 1024 * kBigPer;  // big tiles per step (SDFIBM_ERR_CAPACITY beyond)
constexpr int kBigChunk = 1024;      // default candidate entries per chunk of k_big_force (the autotuner's choice)
constexpr int kBigUPB = 256;         // units, and vertex words, per block (a thread each)
constexpr int kBigStageX = 1024;     // tile x coordinates staged in LDS by k_big_vertices

struct BigMeta {
    int solid;
    int first;       // lowest tile-local index of a cell with an inside vertex (INT_MAX: none)
    long long woff;  // first 64-bit word of its vertex bits
    long long uoff;  // first unit
    int chunk0;      // first chunk of its candidate entries
    int nchunk;
    int ublk0;       // first unit block (kBigUPB units each)
    int nublk;
    int vblk0;       // first vertex-word block
    int pad;
};

// Totals of the step's big tiles: [0] big solids, [3] vertex words, [4] chunks, [5]
// vertex words needed (for the host's buffer growth; the units are fewer), [6] chunks
// needed, [7] unit blocks, [8] vertex-word blocks
constexpr int kBigTotN = 10;

// b with base[b] <= t < base[b + 1] (base ascending, n entries, base[0] = 0)
template <class F>
__device__ inline int big_find(int n, long long t, F base) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (base(mid) <= t)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Words of a vertex row, units of a cell row, and their numbers in the tile.
__host__ __device__ inline int big_vwords(int n0) { return (n0 + 64) >> 6; }
__host__ __device__ inline int big_segs(int n0) { return (n0 + 63) >> 6; }
__device__ inline int big_words(const TileInfo& T) { return (T.n[1] + 1) * (T.n[2] + 1) * big_vwords(T.n[0]); }
__device__ inline int big_units(const TileInfo& T) { return T.n[1] * T.n[2] * big_segs(T.n[0]); }

// Layout of the step's big tiles: one workgroup of 1024 threads, rounds of a solid
// per thread, exclusive scans of vertex words, units and their blocks.
__global__ void __launch_bounds__(1024) k_big_layout(int ns, const TileInfo* __restrict__ Ts,
                                                     const int* __restrict__ qmeta, const int* __restrict__ qlist,
                                                     BigMeta* __restrict__ meta, long long* __restrict__ tot,
                                                     long long word_cap, int* __restrict__ err) {
    __shared__ long long part[4][16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int nbig = qmeta[4];
    if (nbig > kBigMaxSolids) {
        if (tid == 0) atomicOr(err, EF_CODECAP);
        nbig = 0;
    }
    long long carry[4] = {0, 0, 0, 0};
    for (int base = 0; base < nbig; base += 1024) {
        const int b = base + tid;
        long long v[4] = {0, 0, 0, 0};
        int solid = 0;
        if (b < nbig) {
            solid = qlist[4LL * ns + b];
            const TileInfo T = Ts[solid];
            v[0] = big_words(T);
            v[1] = big_units(T);
            v[2] = (v[1] + kBigUPB - 1) / kBigUPB;
            v[3] = (v[0] + kBigUPB - 1) / kBigUPB;
        }
        long long x[4];
        for (int r = 0; r < 4; ++r) {
            x[r] = v[r];
            for (int d = 1; d < 64; d <<= 1) {
                const long long y = __shfl_up(x[r], d, 64);
                if (lane >= d) x[r] += y;
            }
            if (lane == 63) part[r][wv] = x[r];
        }
        __syncthreads();
        long long o[4];
        for (int r = 0; r < 4; ++r) {
            o[r] = carry[r] + x[r] - v[r];
            for (int w = 0; w < 16; ++w) {
                const long long t = part[r][w];
                if (w < wv) o[r] += t;
                carry[r] += t;
            }
        }
        if (b < nbig) meta[b] = BigMeta{solid, 0x7fffffff, o[0], o[1], 0, 0, (int)o[2], (int)v[2], (int)o[3], 0};
        __syncthreads();
    }
    if (tid == 0) {
        // units are at most the vertex words; a solid has at most one partly filled unit block
        const bool fits = carry[0] <= word_cap;
        if (!fits) atomicOr(err, EF_CODECAP);
        tot[0] = fits ? nbig : 0;
        tot[3] = tot[5] = carry[0];
        tot[7] = fits ? carry[2] : 0;
        tot[8] = fits ? carry[3] : 0;
    }
}

// A CSG solid's shape constants copied to LDS for one workgroup iteration (the
// whole workgroup; its previous readers are done first): read from there, they
// are not loaded again after each of the loop's stores, which the compiler
// cannot tell apart from the global table.
__device__ inline void big_csg_to_lds(SolidK& K, CsgK& sh, int tid, int nt) {
    if (K.shape != SDFIBM_SHAPE_CSG) return;  // uniform
    __syncthreads();
    const unsigned* src = reinterpret_cast<const unsigned*>(K.csg);
    unsigned* dst = reinterpret_cast<unsigned*>(&sh);
    for (int t = tid; t < (int)(sizeof(CsgK) / 4); t += nt) dst[t] = src[t];
    __syncthreads();
    K.csg = &sh;
}

// Strict inside test at every big-tile vertex (FP64, the reference's operation
// order where it decides), kBigUPB bit words of one solid per workgroup
// iteration.  Rectilinear meshes, shapes with row intervals: a thread per word
// (row_inside_bits, row_csg_bits; the tile's x coordinates staged in LDS);
// otherwise a wave per word, a vertex per lane, one ballot.  50 CSG solids of
// 40-80 cells: 151 us testing every vertex.
template <int MK>
__global__ void __launch_bounds__(256) k_big_vertices(MeshDev m, const SolidK* __restrict__ Ks,
                                                      const TileInfo* __restrict__ Ts, const BigMeta* __restrict__ meta,
                                                      const long long* __restrict__ tot,
                                                      unsigned long long* __restrict__ vbits) {
    __shared__ CsgK sh_csg;
    __shared__ double sx[MK == MK_RECT ? kBigStageX : 1];
    const int nbig = (int)tot[0];
    const long long nvb = tot[8];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (long long blk = blockIdx.x; blk < nvb; blk += gridDim.x) {
        const int b = big_find(nbig, blk, [&](int x) { return (long long)meta[x].vblk0; });  // uniform
        const BigMeta M = meta[b];
        const TileInfo T = Ts[M.solid];
        SolidK K = Ks[M.solid];
        big_csg_to_lds(K, sh_csg, threadIdx.x, 256);
        const int VX = T.n[0] + 1, VY = T.n[1] + 1, W = big_vwords(T.n[0]), words = big_words(T);
        const float rW = 1.0f / (float)W, rvy = 1.0f / (float)VY;
        const int w0 = (int)(blk - M.vblk0) * kBigUPB, w1 = min(words, w0 + kBigUPB);
        if (MK == MK_RECT && (row_quadric(K.shape) || row_csg(K.shape))) {
            const double* xs = m.xs + T.lo[0];
            if (VX <= kBigStageX) {
                __syncthreads();  // the iteration before has read them
                for (int t = threadIdx.x; t < VX; t += 256) sx[t] = xs[t];
                __syncthreads();
                xs = sx;
            }
            const int w = w0 + (int)threadIdx.x;
            if (w < w1) {
                int r, seg, vj, vk;
                divmod_small(w, W, rW, r, seg);
                divmod_small(r, VY, rvy, vk, vj);
                const double y = m.ys[T.lo[1] + vj], z = m.zs[T.lo[2] + vk];
                const int n = min(64, VX - 64 * seg);
                vbits[M.woff + w] = row_quadric(K.shape) ? row_inside_bits(K, xs + 64 * seg, n, y, z)
                                                         : row_csg_bits(K, xs + 64 * seg, n, y, z);
            }
            continue;
        }
        for (int w = w0 + wv; w < w1; w += 4) {  // wave-uniform
            int r, seg, vj, vk;
            divmod_small(w, W, rW, r, seg);
            divmod_small(r, VY, rvy, vk, vj);
            const int vi = 64 * seg + lane;
            bool in = false;
            if (vi < VX) in = inside_world(K, vertex_pos<MK>(m, T.lo[0] + vi, T.lo[1] + vj, T.lo[2] + vk));
            const unsigned long long bal = __ballot(in);
            if (lane == 0) vbits[M.woff + w] = bal;
        }
    }
}

// Unit u of a tile: its row (j, k), segment, first cell i0, length and first tile
// index.  A unit holds the cells 64 seg .. of its row; rows in index order, so
// consecutive units hold consecutive tile cells.
struct BigUnit {
    int j, k, seg, i0, len, q0;
};
__device__ inline BigUnit big_unit(const TileInfo& T, int u) {
    const int nseg = big_segs(T.n[0]);
    int r;
    BigUnit U;
    divmod_small(u, nseg, 1.0f / (float)nseg, r, U.seg);
    divmod_small(r, T.n[1], 1.0f / (float)T.n[1], U.k, U.j);
    U.i0 = U.seg << 6;
    U.len = min(64, T.n[0] - U.i0);
    U.q0 = r * T.n[0] + U.i0;
    return U;
}

// Iterates the unit blocks of the step's big tiles, one workgroup iteration per
// block (the block's solid found once, uniform): f(b, meta, tile, block, first
// unit of the block, units of the tile).
template <class F>
__device__ inline void big_unit_blocks(const BigMeta* meta, const TileInfo* Ts, const long long* tot, long long code_cap,
                                       F f) {
    const int nbig = (int)tot[0];
    const long long nblk = tot[7];
    for (long long blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const int b = big_find(nbig, blk, [&](int x) { return (long long)meta[x].ublk0; });
        const BigMeta M = meta[b];
        const TileInfo T = Ts[M.solid];
        if (T.off + (long long)T.n[0] * T.n[1] * T.n[2] > code_cap) continue;  // flagged by the tile offsets
        f(b, M, T, blk, (int)(blk - M.ublk0) * kBigUPB, big_units(T));
    }
}

// First cells of the runs of a mask, and the first cell of the run that holds bit p.
__device__ inline unsigned long long run_starts(unsigned long long a) { return a & ~(a << 1); }
__device__ inline int run_start_of(unsigned long long a, int p) {
    return 63 - __builtin_clzll(run_starts(a) & ((2ull << p) - 1ull));
}

// Per unit: its masks from the four vertex rows (j, k) .. (j + 1, k + 1) -- cell i's
// vertices are i and i + 1 of each -- a label at the first cell of each of its
// runs, and the lowest active cell of the solid (one atomic per wave).
__global__ void __launch_bounds__(256) k_big_units(const TileInfo* __restrict__ Ts, BigMeta* __restrict__ meta,
                                                   const long long* __restrict__ tot,
                                                   const unsigned long long* __restrict__ vbits,
                                                   unsigned long long* __restrict__ uact,
                                                   unsigned long long* __restrict__ uall, int* __restrict__ cand,
                                                   long long code_cap) {
    big_unit_blocks(meta, Ts, tot, code_cap, [&](int b, const BigMeta& M, const TileInfo& T, long long, int u0, int units) {
        const int u = u0 + (int)threadIdx.x;
        int lowest = 0x7fffffff;
        if (u < units) {
            const BigUnit U = big_unit(T, u);
            const int W = big_vwords(T.n[0]);
            const unsigned long long* w = vbits + M.woff + U.seg;
            const long long r00 = (long long)W * (U.j + (long long)(T.n[1] + 1) * U.k), r10 = r00 + W;
            const long long r01 = r00 + (long long)W * (T.n[1] + 1), r11 = r01 + W;
            const unsigned long long p = w[r00], q = w[r10], r = w[r01], s = w[r11];
            unsigned long long hiO = 0, hiA = 0;  // vertex 64: the upper vertex of cell 63
            if (U.len == 64) {  // vertex i0 + 64 <= n0: the next word of each row
                const unsigned long long x = w[r00 + 1], y = w[r10 + 1], z = w[r01 + 1], t = w[r11 + 1];
                hiO = (x | y | z | t) << 63;
                hiA = (x & y & z & t) << 63;
            }
            const unsigned long long valid = bits_below(U.len), O = p | q | r | s, A = p & q & r & s;
            const unsigned long long act = (O | (O >> 1) | hiO) & valid;
            uact[M.uoff + u] = act;
            uall[M.uoff + u] = A & ((A >> 1) | hiA) & valid;
            int* L = cand + T.off + U.q0;
            for (unsigned long long st = run_starts(act); st; st &= st - 1ull) {
                const int i = __builtin_ctzll(st);
                L[i] = U.q0 + i;
            }
            if (act) lowest = U.q0 + __builtin_ctzll(act);
        }
        for (int off = 32; off >= 1; off >>= 1) lowest = min(lowest, __shfl_xor(lowest, off, 64));
        if ((threadIdx.x & 63) == 0 &&
            lowest < __hip_atomic_load(&meta[b].first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&meta[b].first, lowest);
    });
}

// The overlaps of unit u's runs with those of the units along +y, +z and -- at the
// unit's end -- +x: f(first cell of the one run, first cell of the other), once
// per pair of overlapping runs and direction.
template <class F>
__device__ inline void big_overlaps(const TileInfo& T, const BigUnit& U, int u, const unsigned long long* act, F f) {
    const unsigned long long A = act[u];
    if (!A) return;
    const int nseg = big_segs(T.n[0]);
    auto side = [&](int v, int dq) {
        const unsigned long long B = act[v];
        for (unsigned long long s = run_starts(A & B); s; s &= s - 1ull) {
            const int p = __builtin_ctzll(s);
            f(U.q0 + run_start_of(A, p), U.q0 + dq + run_start_of(B, p));
        }
    };
    if (U.j + 1 < T.n[1]) side(u + nseg, T.n[0]);
    if (U.k + 1 < T.n[2]) side(u + nseg * T.n[1], T.n[0] * T.n[1]);
    if (U.seg + 1 < nseg && (A >> 63) && (act[u + 1] & 1ull)) f(U.q0 + run_start_of(A, 63), U.q0 + 64);
}

// Unions of overlapping runs.  Bound by the finds' dependent loads: 150 us for 50 CSG
// solids of 40-80 cells with plain finds, 111 with paths halved on the way.
__global__ void __launch_bounds__(256) k_big_hook(const TileInfo* __restrict__ Ts, const BigMeta* __restrict__ meta,
                                                  const long long* __restrict__ tot,
                                                  const unsigned long long* __restrict__ uact, int* cand,
                                                  long long code_cap) {
    big_unit_blocks(meta, Ts, tot, code_cap, [&](int, const BigMeta& M, const TileInfo& T, long long, int u0, int units) {
        const int u = u0 + (int)threadIdx.x;
        if (u >= units) return;
        int* L = cand + T.off;
        big_overlaps(T, big_unit(T, u), u, uact + M.uoff, [&](int x, int y) { uf_unite(L, x, y); });
    });
}

__global__ void __launch_bounds__(256) k_big_compress(const TileInfo* __restrict__ Ts, const BigMeta* __restrict__ meta,
                                                      const long long* __restrict__ tot,
                                                      const unsigned long long* __restrict__ uact, int* cand,
                                                      long long code_cap) {
    big_unit_blocks(meta, Ts, tot, code_cap, [&](int, const BigMeta& M, const TileInfo& T, long long, int u0, int units) {
        const int u = u0 + (int)threadIdx.x;
        if (u >= units) return;
        int* L = cand + T.off;
        const int q0 = big_unit(T, u).q0;
        for (unsigned long long st = run_starts(uact[M.uoff + u]); st; st &= st - 1ull) {
            const int q = q0 + __builtin_ctzll(st);
            L[q] = uf_find(L, q);
        }
    });
}

// Per unit the cells of its runs in the seed's component; ucnt[u] = the ALL_INSIDE
// and cut cells of the units before it in its block, bcnt[block] = the block's
// totals.  Overlapping runs with different labels raise EF_LABEL.
__global__ void __launch_bounds__(256) k_big_reach(const MeshDev m, const TileInfo* __restrict__ Ts,
                                                   const BigMeta* __restrict__ meta, const long long* __restrict__ tot,
                                                   const unsigned long long* __restrict__ uact,
                                                   const unsigned long long* __restrict__ uall,
                                                   unsigned long long* __restrict__ ureach, int2* __restrict__ ucnt,
                                                   const int* __restrict__ cand, int2* __restrict__ bcnt,
                                                   long long code_cap, int* __restrict__ err) {
    __shared__ int scan_lds[32];
    big_unit_blocks(meta, Ts, tot, code_cap, [&](int, const BigMeta& M, const TileInfo& T, long long blk, int u0, int units) {
        const int* L = cand + T.off;
        const unsigned long long* act = uact + M.uoff;
        // the seed: the nearest cell when it has an inside vertex, else the lowest such cell
        // (the first of its run)
        int lseed = -2;
        if (T.seed >= 0) {
            const int si = T.seed % m.nx, sj = (T.seed / m.nx) % m.ny, sk = T.seed / (m.nx * m.ny);
            const int li = si - T.lo[0], lj = sj - T.lo[1], lk = sk - T.lo[2];
            if (li >= 0 && li < T.n[0] && lj >= 0 && lj < T.n[1] && lk >= 0 && lk < T.n[2]) {
                const int r = lj + T.n[1] * lk;
                const unsigned long long a = act[r * big_segs(T.n[0]) + (li >> 6)];
                if ((a >> (li & 63)) & 1ull) lseed = L[r * T.n[0] + (li & ~63) + run_start_of(a, li & 63)];
            }
        }
        if (lseed == -2 && M.first != 0x7fffffff) lseed = L[M.first];
        const int u = u0 + (int)threadIdx.x;
        unsigned long long reach = 0ull, all = 0ull;
        if (u < units) {
            const BigUnit U = big_unit(T, u);
            const unsigned long long a = act[u];
            for (unsigned long long st = run_starts(a); st; st &= st - 1ull) {
                const unsigned long long one = st & (~st + 1ull);
                if (L[U.q0 + __builtin_ctzll(st)] == lseed) reach |= a & ~(a + one);  // the run that starts there
            }
            big_overlaps(T, U, u, act, [&](int x, int y) {
                if (L[x] != L[y]) atomicOr(err, EF_LABEL);
            });
            all = reach & uall[M.uoff + u];
            ureach[M.uoff + u] = reach;
        }
        const int na = __popcll(all), nc = __popcll(reach & ~all);
        int pa, pc, ta, tc;
        block_exscan2<256>(na, nc, pa, pc, ta, tc, scan_lds);
        if (u < units) ucnt[M.uoff + u] = make_int2(pa, pc);
        if (threadIdx.x == 0) bcnt[blk] = make_int2(ta, tc);
        __syncthreads();  // scan_lds is reused by the next block
    });
}

// Per big solid (one workgroup each, one wave: it runs beside the small tiles' kernels,
// where 256 threads waited for room, 160 against 10 us): its unit blocks' counts scanned in order ->
// each block's list offsets (ALL_INSIDE, cut), the solid's two counts and its
// number of candidate chunks.
__global__ void __launch_bounds__(64) k_big_scan(const TileInfo* __restrict__ Ts, BigMeta* __restrict__ meta,
                                                   const long long* __restrict__ tot, const int2* __restrict__ bcnt,
                                                   int2* __restrict__ boff, int2* __restrict__ ncand,
                                                   long long code_cap, int chunk_entries) {
    __shared__ int scan_lds[32];
    const int nbig = (int)tot[0];
    for (int b = blockIdx.x; b < nbig; b += gridDim.x) {
        const BigMeta M = meta[b];
        const TileInfo T = Ts[M.solid];
        if (T.off + (long long)T.n[0] * T.n[1] * T.n[2] > code_cap) continue;  // flagged; uniform
        int ca = 0, cc = 0;  // carries over rounds of 64 blocks
        for (int base = 0; base < M.nublk; base += 64) {
            const int t = base + (int)threadIdx.x;
            const int2 v = t < M.nublk ? bcnt[M.ublk0 + t] : make_int2(0, 0);
            int pa, pc, ta, tc;
            block_exscan2<64>(v.x, v.y, pa, pc, ta, tc, scan_lds);
            if (t < M.nublk) boff[M.ublk0 + t] = make_int2(ca + pa, cc + pc);
            ca += ta;
            cc += tc;
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            ncand[M.solid] = make_int2(ca, cc);
            meta[b].nchunk = (ca + cc + chunk_entries - 1) / chunk_entries;
        }
    }
}

// Codes and candidate lists of the big tiles (ALL_INSIDE cells first, then cut
// cells, each ascending; tile-local linear indices): a wave per unit, a lane per
// cell.  The labels in the list buffer have been read by now.
template <class R>
__global__ void __launch_bounds__(256) k_big_write(const TileInfo* __restrict__ Ts, const BigMeta* __restrict__ meta,
                                                   const long long* __restrict__ tot,
                                                   const unsigned long long* __restrict__ ureach,
                                                   const unsigned long long* __restrict__ uall,
                                                   const int2* __restrict__ ucnt, const int2* __restrict__ boff,
                                                   const int2* __restrict__ ncand, R* __restrict__ codes,
                                                   int* __restrict__ cand, long long code_cap) {
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    big_unit_blocks(meta, Ts, tot, code_cap, [&](int, const BigMeta& M, const TileInfo& T, long long blk, int u0, int units) {
        const int2 o = boff[blk];
        const int n_in = ncand[M.solid].x;
        const unsigned long long below = (1ull << lane) - 1ull;
        for (int u = u0 + wv; u < min(units, u0 + kBigUPB); u += 4) {
            const BigUnit U = big_unit(T, u);
            const unsigned long long reach = ureach[M.uoff + u], all = reach & uall[M.uoff + u], cut = reach & ~all;
            const int2 p = ucnt[M.uoff + u];
            if (lane >= U.len) continue;
            const int q = U.q0 + lane;
            const bool is_all = (all >> lane) & 1ull, is_cut = (cut >> lane) & 1ull;
            if (!is_cut) codes[T.off + q] = is_all ? R(__builtin_huge_val()) : code_none<R>();
            if (is_all) cand[T.off + o.x + p.x + __popcll(all & below)] = q;
            if (is_cut) cand[T.off + n_in + o.y + p.y + __popcll(cut & below)] = q;
        }
    });
}

// Chunk offsets (one workgroup, exclusive scan over the big solids).
__global__ void __launch_bounds__(1024) k_big_chunks(BigMeta* __restrict__ meta, long long* __restrict__ tot,
                                                     long long chunk_cap, int* __restrict__ err) {
    __shared__ int part[1024];
    const int nbig = (int)tot[0];
    const int tid = threadIdx.x;
    int c[kBigPer], sum = 0;
    for (int u = 0; u < kBigPer; ++u) {
        const int b = tid * kBigPer + u;
        c[u] = b < nbig ? meta[b].nchunk : 0;
        sum += c[u];
    }
    part[tid] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int a = tid >= off ? part[tid - off] : 0;
        __syncthreads();
        part[tid] += a;
        __syncthreads();
    }
    int o = part[tid] - sum;
    for (int u = 0; u < kBigPer; ++u) {
        const int b = tid * kBigPer + u;
        if (b < nbig) meta[b].chunk0 = o;
        o += c[u];
    }
    if (tid == 1023) {
        const long long total = part[1023];
        tot[6] = total;
        if (total > chunk_cap) {
            atomicOr(err, EF_CODECAP);
            tot[4] = 0;
        } else {
            tot[4] = total;
        }
    }
}

// Fractions, codes and forcing of one chunk of a big solid's candidates per
// workgroup iteration; FP64 partial force/torque per chunk.
template <class R, int MK, int NT>
__global__ void __launch_bounds__(NT) k_big_force(MeshDev m, const SolidK* __restrict__ Ks,
                                                  const TileInfo* __restrict__ Ts, const BigMeta* __restrict__ meta,
                                                  const long long* __restrict__ tot, const int* __restrict__ cand,
                                                  const int2* __restrict__ ncand, const R* __restrict__ Ux,
                                                  const R* __restrict__ Uy, const R* __restrict__ Uz,
                                                  R* __restrict__ codes, long long code_cap, double dt,
                                                  double* __restrict__ part, int chunk_entries) {
    __shared__ double red[6 * 16];
    __shared__ CsgK sh_csg;
    const int nbig = (int)tot[0];
    const long long nch = tot[4];
    const double dtINV = 1.0 / dt;
    const int tid = threadIdx.x;
    for (long long ch = blockIdx.x; ch < nch; ch += gridDim.x) {
        const int b = big_find(nbig, ch, [&](int x) { return (long long)meta[x].chunk0; });
        const int s = meta[b].solid;
        const TileInfo T = Ts[s];
        if (T.off + (long long)T.n[0] * T.n[1] * T.n[2] > code_cap) continue;  // flagged; uniform per workgroup
        SolidK K = Ks[s];
        big_csg_to_lds(K, sh_csg, tid, NT);
        const int2 cnt = ncand[s];
        const int nin = cnt.x, ntot = cnt.x + cnt.y;
        const int e0 = (int)(ch - meta[b].chunk0) * chunk_entries, e1 = min(e0 + chunk_entries, ntot);
        const int* tl = cand + T.off;
        R* tcodes = codes + T.off;
        const float rn0 = 1.0f / (float)T.n[0], rn1 = 1.0f / (float)T.n[1];
        double acc[6] = {0, 0, 0, 0, 0, 0};
        // the shape known at compile time where it pays (as k_cells' loops)
        auto cells = [&](auto sh) {
            constexpr int SH = decltype(sh)::value;
            SolidK S = K;
            if constexpr (SH >= 0) S.shape = SH;
            for (int e = e0 + tid; e < e1; e += NT) {
                const int q = tl[e];
                int r, i, j, k;
                divmod_small(q, T.n[0], rn0, r, i);
                divmod_small(r, T.n[1], rn1, k, j);
                cell_force<R, MK>(m, S, T.lo[0] + i, T.lo[1] + j, T.lo[2] + k, e >= nin, Ux, Uy, Uz, tcodes + q, dtINV,
                                  acc);
            }
        };
        if (K.shape == SDFIBM_SHAPE_CSG)  // uniform
            cells(std::integral_constant<int, SDFIBM_SHAPE_CSG>{});
        else
            cells(std::integral_constant<int, -1>{});
        block_reduce<6>(acc, red);
        if (tid == 0)
            for (int t = 0; t < 6; ++t) part[6 * ch + t] = acc[t];
    }
}

// Force and torque of the big solids: chunk partials in a fixed order (lanes
// strided over the chunks, then a shuffle tree), x rho_f.
__global__ void __launch_bounds__(256) k_big_ft(const BigMeta* __restrict__ meta, const long long* __restrict__ tot,
                                                const double* __restrict__ part, double rho_f,
                                                double* __restrict__ ft) {
    const int nbig = (int)tot[0];
    const bool ok = tot[4] > 0 || tot[6] == 0;  // chunk partials exist (or there are no candidates)
    const int lane = threadIdx.x & 63;
    const int nw = gridDim.x * (blockDim.x >> 6);
    // a wave per solid: lanes strided over its chunks in order, then a fixed shuffle tree
    for (int b = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); b < nbig; b += nw) {
        const BigMeta M = meta[b];
        double a[6] = {0, 0, 0, 0, 0, 0};
        if (ok)
            for (int c = lane; c < M.nchunk; c += 64)
                for (int t = 0; t < 6; ++t) a[t] += part[6LL * (M.chunk0 + c) + t];
        for (int off = 32; off >= 1; off >>= 1)
            for (int t = 0; t < 6; ++t) a[t] += __shfl_xor(a[t], off, 64);
        if (lane == 0)
            for (int t = 0; t < 6; ++t) ft[6 * M.solid + t] = a[t] * rho_f;
    }
}
