// fused_kernels.hpp -- two AA steps per launch on a periodic D3Q19 box (temporal blocking).
//
// The AA pattern's even step is local (a cell reads and writes its own slots) and its odd step
// reads and writes the neighbours' slots.  Fusing an even step with the following odd step lets
// the even step's post-collision populations stay on chip: a block owns a TX x TY tile of
// (x, y) columns plus a one-cell ring around it, marches up a chunk of z planes and, per plane,
//
//   1. runs the even step of plane p+1 on every cell of tile + ring (loads from `src`),
//   2. publishes to LDS what the odd step of plane p reads: the c_z = -1 populations of plane
//      p+1, the c_z = 0 populations of plane p and the c_z = +1 populations of plane p-1 (each
//      thread keeps its own column's later-needed populations in registers until then),
//   3. runs the odd step of plane p on the tile cells, gathering population v from the LDS copy
//      of cell x - c_v, and pushes its post-collision populations to `dst` at x + c_v.
//
// The ring costs a second even step on (TX+2)(TY+2)/(TX TY) - 1 of the cells and their reads.
// In return each cell is read once and written once per two steps instead of twice each, so
// the HBM traffic per two steps falls from 4 Q s to about (1 + ring) Q s + Q s bytes per cell.
// The odd step's pushes cross tile borders, so `dst` is a second population array: two
// launches in a row go src -> dst -> src.  Both arrays hold the state in the layout the even
// step reads (every cell's pre-collision populations in its own slots), which is the layout of
// a grid after a neighbour step (odd parity); a run from even parity takes one single
// neighbour step first.
//
// Every cell update is the same code as k_aa_periodic's (make_collider and the pair-wise
// collision), and the even step's populations go through the storage type S on the way through
// LDS, as they would through HBM, so in FP64 and FP32-shifted storage the result is bit for bit
// that of an even launch followed by an odd launch.  (In FP16 storage the compiler may round a
// collision's last FMA straight to half in one kernel and through float in the other: the two
// then differ by one unit in the last place of the stored half.)
#pragma once

#include "aa_kernels.hpp"

namespace lumagpu {

template <int TX, int TY>
struct FuseTile {
    static constexpr int WX = TX + 2, WY = TY + 2, C = WX * WY;
};

// Linear block id -> tile id such that the blocks one XCD receives (ids congruent mod 8 under the
// round-robin dispatch) take consecutive tiles: neighbouring tiles, whose ring rows overlap,
// then run on the same XCD and share its L2.
__device__ __forceinline__ int fused_tile_of(int b, int nblocks) {
    const int q = nblocks / 8, r = nblocks % 8, x = b % 8;   // the first r XCDs take one more
    return x * q + (x < r ? x : r) + b / 8;
}

// The 16 populations with a component in x or y, which the odd step takes from other columns
// (the other three, c = (0, 0, +-1) and the rest population, come from the thread's own column).
template <int V>
constexpr int lateral_index() {
    using L = Lattice<19>;
    int k = 0;
    for (int w = 0; w < V; ++w)
        if (L::c(w, 0) != 0 || L::c(w, 1) != 0) ++k;
    return (L::c(V, 0) != 0 || L::c(V, 1) != 0) ? k : -1;
}

// PF: the loads of plane p + 2 are issued at the start of plane p's iteration, into a second
// register set, so they arrive while plane p + 1's even step and plane p's odd step compute
// (one plane of load latency hidden per iteration instead of none).
// WIN: the LDS copy holds, per lateral population v, only the TX x TY window the tile reads
// (the value cell x + c_v of the tile pulls, stored at that cell's index): 16 * TX * TY values
// instead of 19 * (TX + 2)(TY + 2), so two copies of a 32 x 16 tile take 64 KiB and two blocks
// fit a CU; the odd step's LDS reads are then contiguous across the wave.
// MASK: any extents (tiles at the far x and y sides are cut) and a bitmap of the cells the odd step
// takes (deep, see k_deep_bits; null: all).  The even step runs on every cell of tile and ring; what
// it makes of a cell that is not a plain one is read by no deep cell.
// FORCED: a set force field (force_xyz at every cell, zero where the field is): the even step of
// a cell loads it, the odd step takes it from registers.
template <class P, int TX, int TY, bool STORE, bool DB, bool O32 = false, bool PF = false, bool WIN = false,
          bool MASK = false, bool FORCED = false>
__global__ __launch_bounds__((TX + 2) * (TY + 2)) void k_aa_fused2(StepArgs a, void *dst_v, int zc,
                                                                   const uint32_t *deep) {
    using L = Lattice<19>;
    using S = typename P::S;
    using T = typename P::T;
    constexpr int Q = 19;
    constexpr int WX = FuseTile<TX, TY>::WX, C = FuseTile<TX, TY>::C;
    constexpr int TT = TX * TY;
    static_assert(!WIN || DB, "windowed LDS copies are double-buffered");
    // DB: two LDS copies used alternately, so a plane needs one barrier (between publishing and
    // reading) instead of two
    __shared__ S shm[WIN ? 2 * 16 * TT : (DB ? 2 : 1) * Q * C];

    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int ntx = MASK ? (nx + TX - 1) / TX : nx / TX, nty = MASK ? (ny + TY - 1) / TY : ny / TY;
    const int ntz = (nz + zc - 1) / zc;
    const int tile = fused_tile_of(blockIdx.x, ntx * nty * ntz);
    const int tx = tile % ntx, ty = (tile / ntx) % nty, tz = tile / (ntx * nty);
    const int t = threadIdx.x;
    // threads 0 .. TX*TY-1 take the tile row by row (whole waves, rows aligned to the tile's
    // first x), the rest the ring: the row below, the row above, then the two side columns
    int lx, ly;
    if (t < TX * TY) {
        lx = 1 + t % TX;
        ly = 1 + t / TX;
    } else if (t < TX * TY + WX) {
        lx = t - TX * TY;
        ly = 0;
    } else if (t < TX * TY + 2 * WX) {
        lx = t - TX * TY - WX;
        ly = TY + 1;
    } else {
        const int k = t - TX * TY - 2 * WX;
        lx = (k & 1) ? WX - 1 : 0;
        ly = 1 + (k >> 1);
    }
    const int lc = ly * WX + lx;   // the cell's slot in the LDS copy
    int gx = tx * TX - 1 + lx, gy = ty * TY - 1 + ly;
    // a cut tile ends at the grid's last cell; the cell past it is ring, what lies beyond idles at 0
    const bool inner = t < TX * TY && (!MASK || (gx < nx && gy < ny));
    gx = gx < 0 ? gx + nx : (gx >= nx ? (MASK ? 0 : gx - nx) : gx);
    gy = gy < 0 ? gy + ny : (gy >= ny ? (MASK ? 0 : gy - ny) : gy);
    const int z0 = tz * zc, z1 = min(z0 + zc, nz);

    const S *__restrict__ src = static_cast<const S *>(a.f);
    S *__restrict__ dst = static_cast<S *>(dst_v);
    const size_t ps = a.ps;
    const size_t col = (size_t)gx + (size_t)nx * (size_t)gy;
    const size_t plane = (size_t)nx * (size_t)ny;

    // the 19 populations of plane z of this thread's column, as stored
    auto load = [&](int z, S *raw) {
        const size_t cell = col + plane * (size_t)z;
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            if constexpr (O32)
                raw[v] = *reinterpret_cast<const S *>(reinterpret_cast<const char *>(src + (size_t)v * ps) +
                                                      (uint32_t)((uint32_t)cell * (uint32_t)sizeof(S)));
            else
                raw[v] = src[(size_t)v * ps + cell];
        });
    };
    // even step of a column cell from its loaded populations: post-collision populations in
    // storage precision
    using FM = typename P::M;
    struct Force {
        FM v[3];
    };
    auto load_force = [&](int z) {
        Force F{};
        if constexpr (FORCED) {
            const FM *fx = mv<FM>(a.force);
            const size_t cell = col + plane * (size_t)z;
            F.v[0] = fx[cell];
            F.v[1] = fx[a.ncell + cell];
            F.v[2] = fx[2 * a.ncell + cell];
        }
        return F;
    };
    auto deep_word = [&](int z) -> uint32_t {
        if constexpr (MASK) {
            if (deep) {
                const size_t cell = col + plane * (size_t)z;
                return deep[cell >> 5] >> (cell & 31);
            }
        }
        return 1u;
    };
    auto even_from = [&](const S *raw, const Force &F, S *e) {
        T fin[Q];
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            fin[v] = static_cast<T>(raw[v]);
        });
        typename P::M rho, u[3];
        const auto c = make_collider<Q, P>(fin, FORCED ? F.v : nullptr, a, rho, u);
        static_for<(Q - 1) / 2>([&](auto pc) {
            constexpr int v = 2 * decltype(pc)::value;
            T ov, oo;
            c.template pair<v>(fin[v], fin[v + 1], ov, oo);
            e[v] = static_cast<S>(ov);
            e[v + 1] = static_cast<S>(oo);
        });
        e[Q - 1] = static_cast<S>(c(Q - 1, fin[Q - 1]));
    };
    auto even = [&](int z, S *e, Force &F) {
        S raw[Q];
        load(z, raw);
        F = load_force(z);
        even_from(raw, F, e);
    };
    auto wrapz = [&](int z) { return z < 0 ? z + nz : (z >= nz ? z - nz : z); };

    // own column's populations awaiting publication: c_z = 0 of plane p, c_z = +1 of planes p
    // and p - 1 (indexed by population; only the entries of the matching group are used)
    S rmid[Q], rup[Q], rup_prev[Q];
    Force fcur, fnext{};       // the force at planes p and p + 1
    uint32_t dcur = deep_word(z0);
    {
        S e[Q];
        even(wrapz(z0 - 1), e, fcur);
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            if constexpr (L::c(v, 2) == 1) rup_prev[v] = e[v];
        });
        even(z0, e, fcur);
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            if constexpr (L::c(v, 2) == 1) rup[v] = e[v];
            if constexpr (L::c(v, 2) == 0) rmid[v] = e[v];
        });
    }

    // one plane: the even step of plane p + 1 (its populations loaded into `cur`, or loaded
    // here), publication, the odd step of plane p.  With PF the loads of plane p + 2 go into
    // `nxt` first; the caller alternates two buffers, so no copy ties the loads to the loop end.
    // fe / fl: with PF, the force of plane p + 1 (loaded with `cur`) and where that of plane p + 2 goes
    auto plane_step = [&](int p, const S *cur, S *nxt, const Force &fe, Force &fl) {
        S e[Q];
        const uint32_t dnext = deep_word(wrapz(p + 1));
        if constexpr (PF) {
            // unconditionally (the last plane's load is spare): a branch here would make the
            // wait for `cur` also wait for these loads
            load(wrapz(p + 2), nxt);
            fl = load_force(wrapz(p + 2));
            // keep the loads ahead of the plane's work (the scheduler would otherwise sink them
            // towards their use in the next plane)
            __builtin_amdgcn_sched_barrier(0);
            fnext = fe;
            even_from(cur, fe, e);
        } else {
            even(wrapz(p + 1), e, fnext);
        }
        S *sh = WIN ? shm + (p & 1) * (16 * TT) : (DB ? shm + (p & 1) * (Q * C) : shm);
        if constexpr (!DB) __syncthreads();   // the previous plane's odd step has read the LDS copy
        // the own-column populations of the odd step (WIN): c_z = +1 of plane p - 1, c_z = -1 of
        // plane p + 1, the rest population of plane p
        S own4 = S(0), own5 = S(0), own18 = S(0);
        if constexpr (WIN) {
            own4 = rup_prev[4];
            own5 = e[5];
            own18 = rmid[18];
        }
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            constexpr int cz = L::c(v, 2);
            S val;
            if constexpr (cz == -1) val = e[v];
            if constexpr (cz == 0) {
                val = rmid[v];
                rmid[v] = e[v];
            }
            if constexpr (cz == 1) {
                val = rup_prev[v];
                rup_prev[v] = rup[v];
                rup[v] = e[v];
            }
            if constexpr (!WIN) {
                sh[v * C + lc] = val;
            } else if constexpr (lateral_index<v>() >= 0) {
                // the tile cell that pulls this population from this cell
                const int ix = lx - 1 + L::c(v, 0), iy = ly - 1 + L::c(v, 1);
                if (ix >= 0 && ix < TX && iy >= 0 && iy < TY) sh[lateral_index<v>() * TT + iy * TX + ix] = val;
            }
        });
        __syncthreads();
        if (inner && (dcur & 1u)) {
            T fin[Q];
            static_for<Q>([&](auto vc) {
                constexpr int v = decltype(vc)::value;
                constexpr int cx = L::c(v, 0), cy = L::c(v, 1);
                if constexpr (!WIN) {
                    fin[v] = static_cast<T>(sh[v * C + lc - cy * WX - cx]);
                } else if constexpr (lateral_index<v>() >= 0) {
                    fin[v] = static_cast<T>(sh[lateral_index<v>() * TT + (ly - 1) * TX + (lx - 1)]);
                } else {
                    fin[v] = static_cast<T>(v == 4 ? own4 : (v == 5 ? own5 : own18));
                }
            });
            typename P::M rho, u[3];
            const auto c = make_collider<Q, P>(fin, FORCED ? fcur.v : nullptr, a, rho, u);
            if constexpr (STORE) store_macro<3>(a, col + plane * (size_t)p, rho, u);
            const int xm = gx == 0 ? nx - 1 : gx - 1, xp = gx == nx - 1 ? 0 : gx + 1;
            const int ym = gy == 0 ? ny - 1 : gy - 1, yp = gy == ny - 1 ? 0 : gy + 1;
            const int zm = p == 0 ? nz - 1 : p - 1, zp = p == nz - 1 ? 0 : p + 1;
            auto put = [&](auto vc, T o) {
                constexpr int v = decltype(vc)::value;
                constexpr int cx = L::c(v, 0), cy = L::c(v, 1), cz = L::c(v, 2);
                const int xx = cx == 0 ? gx : (cx > 0 ? xp : xm);
                const int yy = cy == 0 ? gy : (cy > 0 ? yp : ym);
                const int zz = cz == 0 ? p : (cz > 0 ? zp : zm);
                if constexpr (O32)
                    st<P, cx == 0>(elem_at<S, true>(dst + (size_t)v * ps,
                                                    (uint32_t)xx + (uint32_t)nx * ((uint32_t)yy + (uint32_t)ny * (uint32_t)zz)), o);
                else
                    st<P, cx == 0>(dst + (size_t)v * ps + cell_of(xx, yy, zz, nx, ny), o);
            };
            static_for<(Q - 1) / 2>([&](auto pc) {
                constexpr int v = 2 * decltype(pc)::value;
                T ov, oo;
                c.template pair<v>(fin[v], fin[v + 1], ov, oo);
                put(std::integral_constant<int, v>{}, ov);
                put(std::integral_constant<int, v + 1>{}, oo);
            });
            put(std::integral_constant<int, Q - 1>{}, c(Q - 1, fin[Q - 1]));
        }
        if constexpr (FORCED) fcur = fnext;
        dcur = dnext;
    };
    if constexpr (PF) {
        S bufA[Q], bufB[Q];
        load(wrapz(z0 + 1), bufA);
        Force fA = load_force(wrapz(z0 + 1)), fB{};
        // pairs of planes with no branch inside the loop body (a conditional second plane merges
        // a path with bufB's loads still in flight into the loop header, whose wait would then
        // cover every outstanding load and store), then an odd last plane
        const int zp = z0 + ((z1 - z0) & ~1);
        for (int p = z0; p < zp; p += 2) {
            plane_step(p, bufA, bufB, fA, fB);
            plane_step(p + 1, bufB, bufA, fB, fA);
        }
        if (zp < z1) plane_step(zp, bufA, bufB, fA, fB);
    } else {
        Force none{};
        for (int p = z0; p < z1; ++p) plane_step(p, nullptr, nullptr, none, none);
    }
}

// Tile shapes the launcher offers; the grid must be a whole number of tiles in x and y.  Shape
// codes: the tile (0-2), + 8 for two LDS copies, + 16 (with two copies) for loads one plane ahead.
enum FusedShape : int { kFuse64x8 = 0, kFuse32x16 = 1, kFuse128x4 = 2 };

inline bool fused_tile(int shape, int &tx, int &ty) {
    static const int t[3][2] = {{64, 8}, {32, 16}, {128, 4}};
    const int k = shape & 7;
    // tile (0-2), + 8 two LDS copies, + 16 loads one plane ahead, + 32 windowed copies; the
    // last two need the two copies
    if (shape < 0 || shape > 63 || k > 2 || (shape & 4) || ((shape & 48) && !(shape & 8))) return false;
    tx = t[k][0];
    ty = t[k][1];
    return true;
}

inline bool fused_shape_fits(int shape, int nx, int ny) {
    int tx, ty;
    if (!fused_tile(shape, tx, ty)) return false;
    return nx % tx == 0 && ny % ty == 0 && nx >= tx && ny >= ty;
}

template <class P, int TX, int TY, bool DB, bool PF = false, bool WIN = false>
hipError_t launch_fused2_t(const StepArgs &a, void *dst, int zc, bool store, hipStream_t s) {
    const int nblocks = (a.nx / TX) * (a.ny / TY) * ((a.nz + zc - 1) / zc);
    const dim3 g(nblocks), b(FuseTile<TX, TY>::C);
    // planes below 4 GiB: 32-bit byte offsets from each population plane's base
    // (measured at 256^3 FP32, 64x8: 302 us per step against 318 with 64-bit addresses)
    const bool o32 = a.ps * sizeof(typename P::S) < (size_t(1) << 32);
    if (o32) {
        if (store) k_aa_fused2<P, TX, TY, true, DB, true, PF, WIN><<<g, b, 0, s>>>(a, dst, zc, nullptr);
        else k_aa_fused2<P, TX, TY, false, DB, true, PF, WIN><<<g, b, 0, s>>>(a, dst, zc, nullptr);
        return hipGetLastError();
    }
    if (store) k_aa_fused2<P, TX, TY, true, DB, false, PF, WIN><<<g, b, 0, s>>>(a, dst, zc, nullptr);
    else k_aa_fused2<P, TX, TY, false, DB, false, PF, WIN><<<g, b, 0, s>>>(a, dst, zc, nullptr);
    return hipGetLastError();
}

template <class P>
hipError_t launch_fused2_p(int shape, const StepArgs &a, void *dst, int zc, bool store, hipStream_t s) {
    if (!fused_shape_fits(shape, a.nx, a.ny) || zc < 1 || a.nz < 3) return hipErrorInvalidValue;
    switch (shape) {
        case kFuse64x8: return launch_fused2_t<P, 64, 8, false>(a, dst, zc, store, s);
        case kFuse32x16: return launch_fused2_t<P, 32, 16, false>(a, dst, zc, store, s);
        case kFuse128x4: return launch_fused2_t<P, 128, 4, false>(a, dst, zc, store, s);
        default: break;
    }
    // two LDS copies fit the 160 KiB of a CU for storage types up to 4 bytes
    if constexpr (sizeof(typename P::S) <= 4) {
        if (shape == 8 + kFuse64x8) return launch_fused2_t<P, 64, 8, true>(a, dst, zc, store, s);
        if (shape == 8 + kFuse32x16) return launch_fused2_t<P, 32, 16, true>(a, dst, zc, store, s);
        if (shape == 8 + kFuse128x4) return launch_fused2_t<P, 128, 4, true>(a, dst, zc, store, s);
        if (shape == 24 + kFuse64x8) return launch_fused2_t<P, 64, 8, true, true>(a, dst, zc, store, s);
        if (shape == 24 + kFuse32x16) return launch_fused2_t<P, 32, 16, true, true>(a, dst, zc, store, s);
        if (shape == 24 + kFuse128x4) return launch_fused2_t<P, 128, 4, true, true>(a, dst, zc, store, s);
        if (shape == 40 + kFuse64x8) return launch_fused2_t<P, 64, 8, true, false, true>(a, dst, zc, store, s);
        if (shape == 40 + kFuse32x16) return launch_fused2_t<P, 32, 16, true, false, true>(a, dst, zc, store, s);
        if (shape == 56 + kFuse32x16) return launch_fused2_t<P, 32, 16, true, true, true>(a, dst, zc, store, s);
    }
    return hipErrorInvalidValue;
}

// ---- two steps per launch on any D3Q19 grid --------------------------------------------------
// Where the neighbourhood of a cell holds nothing but plain cells (fluid, no boundary source, no
// body force of its own), its two steps need no flag: these deep cells take k_aa_fused2, and the rest,
// a surface, takes two list launches around it, out of the populations `src` into `dst`:
//   1. the even step of the list S1 = S + its neighbours, src -> dst (S: stepped, not deep)
//   2. k_aa_fused2 on the deep cells, src -> dst
//   3. the odd step of S, in place in dst
// A slot belongs, in each of the two layouts, to one cell, which alone reads and writes it.  Step 1
// leaves the even results of S1 in their cells' slots; step 2 writes the slots that deep cells own
// in the odd layout, so it comes after 1 and spares every slot that step 3 reads, since those are
// owned by S.  A slot of neither kind belongs to a solid, forced-equilibrium or other site that
// never steps: it holds what it held (run_pairs copies those after a change of state or labels),
// or what S pushes there.

// deep: plain, and every neighbour plain; with bodies, none of them a support (forced)
// rest: the cells k_aa_masked_list steps that are not deep
template <int Q>
__global__ __launch_bounds__(256) void k_deep_bits(StepArgs a, int bodies, uint32_t *deep, uint32_t *rest) {
    using L = Lattice<Q>;
    const size_t c = (size_t)blockIdx.x * 256 + threadIdx.x;
    bool is_deep = false, is_rest = false;
    if (c < a.ncell) {
        auto plain = [&](size_t k) {
            return ((a.plain[k >> 5] >> (k & 31)) & 1u) && !(bodies && (a.flags[k] & kForcedBit));
        };
        is_deep = plain(c);
        int x, y, z;
        cell_coords(a, (uint32_t)c, x, y, z);
        Nbr nb;
        nb.init(x, y, z, a.nx, a.ny, a.nz);
        for (int v = 0; v < Q - 1 && is_deep; ++v)
            is_deep = plain(nb.at(L::c(v, 0), L::c(v, 1), L::c(v, 2), a.nx, a.ny));
        const unsigned fl = a.flags[c];
        const int t = fl & kTypeMask;
        const bool stepped = t == kFluid || t == kExtrapRight ||
                             (t == kVelocity && a.regularised && ((fl >> kNormalShift) & 7) != kNormalEdge);
        is_rest = stepped && !is_deep;
    }
    const uint64_t d = __ballot(is_deep), r = __ballot(is_rest);
    if ((threadIdx.x & 31) == 0 && c < a.ncell) {
        deep[c >> 5] = (uint32_t)(d >> (threadIdx.x & 32));
        rest[c >> 5] = (uint32_t)(r >> (threadIdx.x & 32));
    }
}
// near: rest and the stepped neighbours of rest (a neighbour of a listed or edge site that steps
// and is not in rest is deep)
template <int Q>
__global__ __launch_bounds__(256) void k_near_bits(StepArgs a, const uint32_t *deep, const uint32_t *rest, uint32_t *near) {
    using L = Lattice<Q>;
    const size_t c = (size_t)blockIdx.x * 256 + threadIdx.x;
    bool in = false;
    if (c < a.ncell) {
        auto bit = [](const uint32_t *m, size_t k) { return ((m[k >> 5] >> (k & 31)) & 1u) != 0; };
        in = bit(rest, c);
        if (!in && bit(deep, c)) {
            int x, y, z;
            cell_coords(a, (uint32_t)c, x, y, z);
            Nbr nb;
            nb.init(x, y, z, a.nx, a.ny, a.nz);
            for (int v = 0; v < Q - 1 && !in; ++v) in = bit(rest, nb.at(L::c(v, 0), L::c(v, 1), L::c(v, 2), a.nx, a.ny));
        }
    }
    const uint64_t m = __ballot(in);
    if ((threadIdx.x & 31) == 0 && c < a.ncell) near[c >> 5] = (uint32_t)(m >> (threadIdx.x & 32));
}

// Tile and z chunk for a grid: one block fits a CU, so the cost is the rounds of 256 blocks times
// the planes each takes, its two of start-up included (an even step without an odd one: counted as
// one), times the tile's cells; 64 x 8 unless its cut tiles cost more than 32 x 16's.
struct PairPlan {
    int shape, zc;
};
inline PairPlan plan_pair(int nx, int ny, int nz) {
    PairPlan best{kFuse64x8, nz};
    double cost = 0.0;
    for (int shape : {kFuse64x8, kFuse32x16}) {
        int tx, ty;
        fused_tile(shape, tx, ty);
        const long tiles = (long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
        for (int n = 1; n <= nz; ++n) {
            const int zc = (nz + n - 1) / n;
            const double rounds = (double)((tiles * ((nz + zc - 1) / zc) + 255) / 256);
            // 32 x 16 moves its rows in halves of the 64 x 8 tile's lines: 1.08 per cell
            const double c = rounds * (zc + 1) * (shape == kFuse64x8 ? 1.0 : 1.08);
            if (cost == 0.0 || c < cost) {
                cost = c;
                best = PairPlan{shape, zc};
            }
        }
    }
    return best;
}

template <class P, int TX, int TY, bool MASK, bool FORCED>
hipError_t launch_pair_t(const StepArgs &a, void *dst, int zc, const uint32_t *deep, bool store, hipStream_t s) {
    const unsigned nb = (unsigned)(((a.nx + TX - 1) / TX) * ((a.ny + TY - 1) / TY) * ((a.nz + zc - 1) / zc));
    const dim3 b(FuseTile<TX, TY>::C);
    const bool o32 = a.ps * sizeof(typename P::S) < (size_t(1) << 32);
    if (!o32) return hipErrorInvalidValue;   // pair_ok keeps such grids on single steps
    if (store) k_aa_fused2<P, TX, TY, true, true, true, true, false, MASK, FORCED><<<nb, b, 0, s>>>(a, dst, zc, deep);
    else k_aa_fused2<P, TX, TY, false, true, true, true, false, MASK, FORCED><<<nb, b, 0, s>>>(a, dst, zc, deep);
    return hipGetLastError();
}

// the deep cells of any grid (deep null: every cell), with or without a set force field
template <class P>
hipError_t launch_pair_p(const StepArgs &a, void *dst, PairPlan pl, const uint32_t *deep, bool forced, bool store,
                         hipStream_t s) {
    const bool whole = !deep && !forced && fused_shape_fits(pl.shape, a.nx, a.ny);
    if (pl.shape == kFuse64x8) {
        if (whole) return launch_pair_t<P, 64, 8, false, false>(a, dst, pl.zc, deep, store, s);
        if (forced) return launch_pair_t<P, 64, 8, true, true>(a, dst, pl.zc, deep, store, s);
        return launch_pair_t<P, 64, 8, true, false>(a, dst, pl.zc, deep, store, s);
    }
    if (whole) return launch_pair_t<P, 32, 16, false, false>(a, dst, pl.zc, deep, store, s);
    if (forced) return launch_pair_t<P, 32, 16, true, true>(a, dst, pl.zc, deep, store, s);
    return launch_pair_t<P, 32, 16, true, false>(a, dst, pl.zc, deep, store, s);
}

}  // namespace lumagpu
