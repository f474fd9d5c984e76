// k_sweep.hip — several Gauss-Seidel sweeps of the pressure per launch
// (gs_solve_kernel, asiroisvigneux/Blaze src/FluidSolver.cu:517-599), each
// workgroup keeping a tile of columns on the chip while it walks the slabs.
//
// Why: one sweep per launch (k_project.hip) moves 12 bytes per cell and
// sweep and, on small grids, is one launch and one latency-bound walk per
// sweep; a walk over the slabs can carry several sweeps at once, because a
// sweep needs of the sweep before it only values up to one slab ahead. In
// step t half sweep h (even: red, odd: black) is at slab group t - h: it
// reads what half sweep h - 1 wrote to LDS in the step before (the other
// colour at its own group) and what half sweep h - 2 wrote one group further
// (its own old values). In x and y the tile's rim is computed again by every
// tile that needs it. Every cell's update is the reference's expression in
// the reference's order on the same values, so the bits are those of the
// one-sweep kernels, whatever the tile.
//
// What bounds it: on small grids the step (LDS reads, one dependent chain of
// four updates, an LDS write, a barrier: about 0.45 us). At 256^3 no one unit:
// of a launch of two sweeps the LDS is busy for 53% (nearly half of that in
// bank conflicts) and the vector units issue for 41%, it moves 5.6 TB/s, and a
// wave waits half of its time. So half sweeps are spread over waves
// (items of 64 columns) rather than walked one after the other by the wave
// that owns a column: the first build of this kernel, a column per lane for
// all sweeps, took 9.8 us per sweep at 128^3 (8x8 columns, 3 sweeps) against
// 6.9. Measured and dropped: two slab groups per step (6.9 against 7.1
// us at 128^3, 20.4 against 28.9 at 256^3), old pressure and rhs 6 or 8
// groups ahead instead of 2 or 4 (no difference), each LDS plane's pitch
// chosen against bank conflicts (5% fewer conflicts in a model of them).
// (These on constant pressure.)
//
// us per sweep on random pressure, best kernel of one sweep per launch -> here
// in calls of 10 (3 + 3 + 2 + 2) / of 120 sweeps:
//   32^3 6.9 -> 3.5 / 2.7, 64^3 10.7 -> 5.0 / 3.8, 90x75x62 11.9 -> 4.9 / 4.3,
//   96^3 14.8 -> 6.7 / 6.0, 128^3 20.6 -> 7.9 / 7.1, 192^3 29.8 -> 15.8 / 13.9,
//   256^3 40.6 -> 23.2 / 22.9, 512^3 388 -> 231 / 253.
// In the solves of the 256^3 explosion 22.7, the events around each call's
// launches included.
#include "solver.h"

namespace blz {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

constexpr float NEG0 = -0.0f;

// Geometry of a BX x BY tile of columns and T sweeps. A cell at L1 distance
// a from the tile matters to the tile's last values as far as the five-point
// update carries it: half sweep h is needed where a <= 2T - 1 - h, the old
// red pressure where a <= 2T - 1, the old black one where a <= 2T. A half
// sweep's columns are cut into items of 64, K of which make a compute wave;
// loader waves fetch the old pressure, P slab groups ahead.
template <int BX, int BY, int T, int K, int P>
struct Tile {
    static constexpr int R = 2 * T;
    static constexpr int RW = BX + 2 * R, RH = BY + 2 * R;
    // LDS planes: 0 old red, 1 old black, h + 2 the values of half sweep h
    // (all but the last), each as large as its columns' bounding box
    static constexpr int PLANES = 2 * T + 1;
    static constexpr int reach(int p) { return p == 0 ? 2 * T - 1 : 2 * T + 1 - p; }
    static constexpr int left(int p) { return (R - reach(p)) >> 1; } // first pair of columns
    static constexpr int pitch(int p) { return ((R + reach(p) + BX - 1) >> 1) - left(p) + 1; }
    static constexpr int cells(int p) { return pitch(p) * (BY + 2 * reach(p)); }
    static constexpr int base(int p) { return p == 0 ? 0 : base(p - 1) + cells(p - 1); }
    static constexpr int SEG = base(PLANES); // cells of one step parity
    static constexpr int cell(int p, int x, int y) {
        return base(p) + (y - (R - reach(p))) * pitch(p) + ((x >> 1) - left(p));
    }
    static constexpr int dist(int x, int y) {
        const int dx = x < R ? R - x : (x >= R + BX ? x - (R + BX - 1) : 0);
        const int dy = y < R ? R - y : (y >= R + BY ? y - (R + BY - 1) : 0);
        return dx + dy;
    }
    static constexpr int columns(int colour, int reach) {
        int n = 0;
        for (int y = 0; y < RH; ++y)
            for (int x = 0; x < RW; ++x) n += ((x + y) & 1) == colour && dist(x, y) <= reach;
        return n;
    }
    static constexpr int items() {
        int n = 0;
        for (int h = 0; h < 2 * T; ++h) n += (columns(h & 1, 2 * T - 1 - h) + 63) / 64;
        return n;
    }
    static constexpr int NI = items();
    static constexpr int CW = (NI + K - 1) / K; // compute waves; wave w has items w, w + CW, ...
    static constexpr int NL = (columns(0, 2 * T - 1) + 63) / 64 + (columns(1, 2 * T) + 63) / 64; // loaders' items
    static constexpr int LMAX = 16 / P;               // items of a loader wave, at most
    static constexpr int LW = (NL + LMAX - 1) / LMAX; // loader waves
    static constexpr int LI = (NL + LW - 1) / LW;     // items of each
    static constexpr int WAVES = CW + LW;
    static constexpr int THREADS = 64 * WAVES;
    static_assert(THREADS <= 1024, "a workgroup has at most 16 waves");
    static_assert(P % 2 == 0, "the LDS parity of a step is that of its place in a round");
    // of an item's lane: column x | y << 6 | in the tile << 12 | used << 13 |
    // half sweep << 14, and the LDS cells of the column's left, right, upper
    // and lower neighbours in the plane the half sweep reads, of its own old
    // values and of its new ones; of a loader's lane x | y << 6 | used << 12
    // | black << 13 and the column's cell
    struct Lane {
        unsigned col;
        unsigned short l, r, n, s, i, o;
    };
    struct Load {
        unsigned short col, o;
    };
    struct Table {
        Lane item[CW * K * 64];
        Load load[LW * LI * 64];
    };
    static constexpr Table make() {
        Table t{};
        int it = 0;
        for (int h = 0; h < 2 * T; ++h) {
            int n = 0;
            for (int y = 0; y < RH; ++y)
                for (int x = 0; x < RW; ++x)
                    if (((x + y) & 1) == (h & 1) && dist(x, y) <= 2 * T - 1 - h) {
                        Lane& e = t.item[64 * it + n];
                        e.col = (unsigned)(x | (y << 6) | ((dist(x, y) == 0 ? 1 : 0) << 12) | (1 << 13) | (h << 14));
                        e.l = (unsigned short)cell(h + 1, x - 1, y);
                        e.r = (unsigned short)cell(h + 1, x + 1, y);
                        e.n = (unsigned short)cell(h + 1, x, y - 1);
                        e.s = (unsigned short)cell(h + 1, x, y + 1);
                        e.i = (unsigned short)cell(h, x, y);
                        e.o = (unsigned short)(h < 2 * T - 1 ? cell(h + 2, x, y) : 0);
                        if (++n == 64) n = 0, ++it;
                    }
            if (n) {
                for (; n < 64; ++n) t.item[64 * it + n] = Lane{(unsigned)(h << 14), 0, 0, 0, 0, 0, 0};
                ++it;
            }
        }
        for (; it < CW * K; ++it) // no item: a half sweep that never comes
            for (int n = 0; n < 64; ++n) t.item[64 * it + n] = Lane{0xfffu << 14, 0, 0, 0, 0, 0, 0};
        int n = 0;
        for (int c = 0; c < 2; ++c) {
            for (int y = 0; y < RH; ++y)
                for (int x = 0; x < RW; ++x)
                    if (((x + y) & 1) == c && dist(x, y) <= 2 * T - 1 + c)
                        t.load[n++] = Load{(unsigned short)(x | (y << 6) | (1 << 12) | (c << 13)),
                                           (unsigned short)cell(c, x, y)};
            for (; n % 64; ++n) t.load[n] = Load{(unsigned short)(c << 13), 0};
        }
        for (; n < LW * LI * 64; ++n) t.load[n] = Load{0, 0};
        return t;
    }
    static constexpr Table table = make();
};

// Division: q0 = num*y, r = fma(-q0, d, num), q = fma(r, y, q0) equals IEEE
// num / d where 2^-125 <= |num| <= FLT_MAX (k_project.hip). q0 +-normal
// implies that range; a q0 of +0 comes from num = +0 or from tiny positive
// numerators whose quotient is +0 as well. A lane whose q0 is of any other
// class sends its wave through IEEE division for the group.
constexpr int BAD_CLASS = 0x3ff & ~((1 << 3) | (1 << 6) | (1 << 8));

// the values a step wrote to LDS are there for the next step's readers;
// loads from global memory stay in flight
__device__ __forceinline__ void step_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct Mem {
    __amdgpu_buffer_rsrc_t rs;
    int gs, Dg; // bytes per slab group, groups
    // group g of the column at byte offset v of its group -1 (groups before
    // the first and past the last: the ghost groups)
    __device__ __forceinline__ f4v load(int v, int g) const {
        const int so = __builtin_amdgcn_readfirstlane(min(max(g + 1, 0), Dg + 1) * gs);
        return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rs, v, so, 0));
    }
};

// 64 columns of one half sweep
template <int P>
struct Item {
    int h;                      // half sweep: at group t - h in step t
    int aL, aR, aN, aS, aI, aO; // LDS cells: the neighbours' values, the column's old and new ones
    int vr, vd;                 // byte offsets of the column (group -1) in the rhs and new pressure planes
    float dm, ym, de, ye;       // neighbour counts and their reciprocals, inside and at the k edges
    bool active, publish, store;
    f4v own;                    // the column's old values of the group
    float pv;                   // its new value of the slab below
    f4v sx[P];                  // rhs loads in flight
};

template <int K, int P, int SEG, int LASTH>
struct Compute {
    Mem m;
    f4v* lds;
    int D;
    float scale;
    Item<P> it[K];

    template <int PAR>
    __device__ __forceinline__ f4v read(int a) const {
        return lds[a + (PAR ^ 1) * SEG];
    }
    template <int PAR>
    __device__ __forceinline__ void put(const Item<P>& e, const f4v& n, int g) {
        if (e.publish) lds[e.aO + PAR * SEG] = n;
        if (e.h >= LASTH - 1 && e.store) // the last red and black half sweeps: the result
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, n), m.rs, e.vd,
                                                   __builtin_amdgcn_readfirstlane((g + 1) * m.gs), 0);
    }

    // the group's updates from v = scale * rhs + the four neighbours. BOUND:
    // slab 0, slab D - 1 or slabs k >= D may be in it; EXACT: IEEE division.
    // false: a lane needs IEEE division.
    template <bool BOUND, bool EXACT>
    __device__ __forceinline__ bool chain(const Item<P>& e, const f4v& v, float next, int g, f4v& n) const {
        const int last = D - 1 - 4 * g; // slab D - 1 counted from the group's first
        float pv = BOUND && g == 0 ? NEG0 : e.pv;
        const f4v up = {e.own[1], e.own[2], e.own[3], BOUND && g == m.Dg - 1 ? NEG0 : next};
        bool bad = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float num = v[k] + pv;
            num = num + up[k];
            const bool edge = BOUND && ((k == 0 && g == 0) | (k == last));
            const float d = edge ? e.de : e.dm;
            float q;
            if constexpr (EXACT) {
                q = num / d;
            } else {
                const float y = edge ? e.ye : e.ym;
                const float q0 = num * y;
                const bool c = __builtin_amdgcn_classf(q0, BAD_CLASS);
                bad |= BOUND ? c & (k <= last) : c;
                const float r = fmaf(-q0, d, num);
                q = fmaf(r, y, q0);
            }
            pv = q;
            n[k] = BOUND && k > last ? NEG0 : q;
        }
        return EXACT || !__builtin_amdgcn_ballot_w64(bad & e.active);
    }

    // the items' reads of a step, all before the first write
    template <int U, int Q>
    __device__ __forceinline__ void gather(f4v (&up)[K], f4v (&v)[K]) const {
        constexpr int PAR = U & 1;
        const Item<P>& e = it[Q];
        const f4v l = read<PAR>(e.aL), r = read<PAR>(e.aR), a = read<PAR>(e.aN), b = read<PAR>(e.aS);
        up[Q] = read<PAR>(e.aI); // the column's old values of the next group
        f4v x = scale * e.sx[U];
        x = x + l;
        x = x + r;
        x = x + a;
        v[Q] = x + b;
        if constexpr (Q + 1 < K) gather<U, Q + 1>(up, v);
    }
    template <int U, int Q>
    __device__ __forceinline__ void update(const f4v (&up)[K], const f4v (&v)[K], int t) {
        constexpr int PAR = U & 1;
        Item<P>& e = it[Q];
        const int g = t - e.h;
        f4v n;
        if (g > 0 && g < m.Dg - 1) {
            if (!chain<false, false>(e, v[Q], up[Q][0], g, n)) (void)chain<false, true>(e, v[Q], up[Q][0], g, n);
            put<PAR>(e, n, g);
            // the two (unlike) comments keep the compiler from merging the
            // paths' last writes into one through a pointer, which would put
            // the item into scratch memory
            asm volatile("; interior group");
        } else if (g >= 0 && g < m.Dg) {
            if (!chain<true, false>(e, v[Q], up[Q][0], g, n)) (void)chain<true, true>(e, v[Q], up[Q][0], g, n);
            put<PAR>(e, n, g);
            asm volatile("; first or last group");
        } else {
            n[3] = NEG0;
        }
        e.sx[U] = m.load(e.vr, g + P);
        e.pv = n[3];
        e.own = up[Q];
        if constexpr (Q + 1 < K) update<U, Q + 1>(up, v, t);
    }
    // steps t .. end - 1 of one round over the loads in flight; U: the
    // step's place in the round
    template <int U>
    __device__ __forceinline__ void round(int t, int end) {
        if constexpr (U < P) {
            if (t + U >= end) return;
            f4v up[K], v[K];
            gather<U, 0>(up, v);
            update<U, 0>(up, v, t + U);
            step_barrier();
            round<U + 1>(t, end);
        }
    }
};

// one round of a loader wave: the old pressure that arrived goes to LDS
template <int U, int P, int LI, int SEG>
__device__ __forceinline__ void load_round(const Mem& m, f4v* lds, const int (&v)[LI], const int (&o)[LI],
                                           const int (&ahead)[LI], const bool (&in)[LI], f4v (&s)[LI][P], int t,
                                           int end) {
    if constexpr (U < P) {
        if (t + U >= end) return;
#pragma unroll
        for (int q = 0; q < LI; ++q) {
            if (in[q]) lds[o[q] + (U & 1) * SEG] = s[q][U];
            s[q][U] = m.load(v[q], t + U + P + ahead[q]);
        }
        step_barrier();
        load_round<U + 1, P, LI, SEG>(m, lds, v, o, ahead, in, s, t, end);
    }
}

// T sweeps of one tile. The walk starts at t = -2 (the old pressure of
// group 0 arrives) and ends with the last half sweep's last group; all waves
// run the same number of steps.
template <int BX, int BY, int T, int K, int P>
__device__ __forceinline__ void sweep_tile(const FusedScene& a, int tile) {
    using G = Tile<BX, BY, T, K, P>;
    __shared__ f4v lds[2 * G::SEG];
    const int ntx = (a.W + BX - 1) / BX;
    const int ty = tile / ntx, tx = tile - ty * ntx;
    const int i0 = tx * BX - G::R, j0 = ty * BY - G::R; // even: x + y has the colour of i + j
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // -0, the identity of the sum, wherever a neighbour may lie outside the grid
    for (int q = threadIdx.x; q < 2 * G::SEG; q += G::THREADS) lds[q] = f4v{NEG0, NEG0, NEG0, NEG0};
    Mem m;
    m.rs = __builtin_amdgcn_make_buffer_rsrc((void*)a.base, (short)0, (int)a.nbytes, 0x00020000);
    m.gs = a.Hp * a.Wp * 16;
    m.Dg = (a.D + 3) >> 2;
    // byte offset of a column in group -1 of a plane; columns outside the
    // grid address one inside, their values go nowhere
    auto offset = [&](int i, int j) {
        i = min(max(i, 0), a.W - 1);
        j = min(max(j, 0), a.H - 1);
        return (unsigned)(16 * ((j + 1) * a.Wp + ((i >> 1) + 1)));
    };
    auto in_grid = [&](int i, int j) { return i >= 0 && i < a.W && j >= 0 && j < a.H; };
    const int end = m.Dg + 2 * T - 1;
    __syncthreads();
    if (w < G::CW) {
        Compute<K, P, G::SEG, 2 * T - 1> c;
        c.m = m;
        c.lds = lds;
        c.D = a.D;
        c.scale = a.scale;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            Item<P>& e = c.it[q];
            const typename G::Lane u = G::table.item[64 * (w + q * G::CW) + lane];
            e.h = __builtin_amdgcn_readfirstlane((int)(u.col >> 14));
            const int i = i0 + (int)(u.col & 63u), j = j0 + (int)((u.col >> 6) & 63u);
            e.active = ((u.col >> 13) & 1u) && in_grid(i, j);
            e.publish = e.active && e.h < 2 * T - 1;
            e.store = e.active && ((u.col >> 12) & 1u);
            e.aL = u.l;
            e.aR = u.r;
            e.aN = u.n;
            e.aS = u.s;
            e.aI = u.i;
            e.aO = u.o;
            e.vr = (int)(((e.h & 1) ? a.rhsB : a.rhsR) + offset(i, j));
            e.vd = (int)(((e.h & 1) ? a.dstB : a.dstR) + offset(i, j));
            const int ic = min(max(i, 0), a.W - 1), jc = min(max(j, 0), a.H - 1);
            const int cnt = (int)(ic > 0) + (int)(ic < a.W - 1) + (int)(jc > 0) + (int)(jc < a.H - 1);
            e.dm = (float)(cnt + 2);
            e.de = (float)(cnt + 1);
            e.ym = 1.0f / e.dm;
            e.ye = 1.0f / e.de;
            e.pv = NEG0;
            e.own = f4v{NEG0, NEG0, NEG0, NEG0};
#pragma unroll
            for (int k = 0; k < P; ++k) e.sx[k] = m.load(e.vr, k - 2 - e.h);
        }
#pragma unroll 1
        for (int t = -2; t < end; t += P) c.template round<0>(t, end);
    } else {
        // loader: in step t old red of group t + 2 and old black of group
        // t + 1 go to LDS
        int v[G::LI], o[G::LI], ahead[G::LI];
        bool in[G::LI];
        f4v s[G::LI][P];
#pragma unroll
        for (int q = 0; q < G::LI; ++q) {
            const typename G::Load u = G::table.load[64 * ((w - G::CW) + q * G::LW) + lane];
            const int i = i0 + (int)(u.col & 63u), j = j0 + (int)((u.col >> 6) & 63u);
            const int black = __builtin_amdgcn_readfirstlane((int)(u.col >> 13));
            ahead[q] = 2 - black;
            v[q] = (int)((black ? a.srcB : a.srcR) + offset(i, j));
            in[q] = ((u.col >> 12) & 1u) && in_grid(i, j);
            o[q] = u.o;
#pragma unroll
            for (int k = 0; k < P; ++k) s[q][k] = m.load(v[q], k - 2 + ahead[q]);
        }
#pragma unroll 1
        for (int t = -2; t < end; t += P) load_round<0, P, G::LI, G::SEG>(m, lds, v, o, ahead, in, s, t, end);
    }
}

// consecutive workgroups go to the eight XCDs in turn: give each XCD one
// run of neighbouring tiles, whose rims then meet in one L2
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int q = nb >> 3, r = nb & 7, c = b & 7;
    return c * q + min(c, r) + (b >> 3);
}

template <int BX, int BY, int T, int K, int P>
__global__ void __launch_bounds__((Tile<BX, BY, T, K, P>::THREADS)) k_rbgs_tile(FusedScene a) {
    if (*a.stop) return; // the solve has converged
    sweep_tile<BX, BY, T, K, P>(a, xcd_tile((int)blockIdx.x, (int)gridDim.x));
}

// the same sweeps over several grids in one launch: block b belongs to the
// last table entry whose first_block <= b
template <int BX, int BY, int T, int K, int P>
__global__ void __launch_bounds__((Tile<BX, BY, T, K, P>::THREADS)) k_rbgs_tile_multi(
    const FusedScene* __restrict__ sc, int n) {
    const int b = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sc[mid].first_block <= b) lo = mid;
        else hi = mid - 1;
    }
    const FusedScene e = sc[lo];
    if (*e.stop) return;
    sweep_tile<BX, BY, T, K, P>(e, b - e.first_block);
}

template <int BX, int BY, int T, int K, int P>
int go(hipStream_t st, const FusedScene* one, const FusedScene* tab, int n, int blocks) {
    const dim3 grid((unsigned)blocks), block(Tile<BX, BY, T, K, P>::THREADS);
    if (one) hipLaunchKernelGGL((k_rbgs_tile<BX, BY, T, K, P>), grid, block, 0, st, *one);
    else hipLaunchKernelGGL((k_rbgs_tile_multi<BX, BY, T, K, P>), grid, block, 0, st, tab, n);
    BLZ_HIP(hipGetLastError());
    return BLZ_OK;
}

// The tiles in use: columns, the most sweeps of a launch, and how many are
// usual. From 16x8 on two, as three need two items per wave: us per sweep of
// two / three per launch on random pressure 144^3 10.0 / 11.0, 192^3 13.9 /
// 16.8, 256^3 22.9 / 23.0; in the 256^3 explosion's solves a launch of two takes
// 42 us and one of three 69. Three win where the planes outgrow the 256 MB
// Infinity Cache (320^3 73 / 63, 512^3 253 / 216).
struct Family {
    int bx, by, tmax, usual;
};
constexpr Family kFamilies[TILE_FAMILIES] = {{4, 4, 5, 4},  {8, 4, 3, 3},  {8, 8, 3, 3},
                                             {16, 8, 3, 2}, {16, 12, 3, 2}, {16, 16, 3, 2}};

// T sweeps with a family's tiles, of one grid or of a table of grids
int tile_sweeps(hipStream_t st, int family, int t, const FusedScene* one, const FusedScene* tab, int n, int blocks) {
    switch (family * 10 + t) {
    case 2: return go<4, 4, 2, 1, 2>(st, one, tab, n, blocks);
    case 3: return go<4, 4, 3, 1, 2>(st, one, tab, n, blocks);
    case 4: return go<4, 4, 4, 1, 2>(st, one, tab, n, blocks);
    case 5: return go<4, 4, 5, 2, 2>(st, one, tab, n, blocks);
    case 12: return go<8, 4, 2, 1, 4>(st, one, tab, n, blocks);
    case 13: return go<8, 4, 3, 1, 4>(st, one, tab, n, blocks);
    case 22: return go<8, 8, 2, 1, 4>(st, one, tab, n, blocks);
    case 23: return go<8, 8, 3, 1, 4>(st, one, tab, n, blocks);
    case 32: return go<16, 8, 2, 1, 4>(st, one, tab, n, blocks);
    case 33: return go<16, 8, 3, 2, 4>(st, one, tab, n, blocks);
    case 42: return go<16, 12, 2, 1, 4>(st, one, tab, n, blocks);
    case 43: return go<16, 12, 3, 2, 2>(st, one, tab, n, blocks);
    case 52: return go<16, 16, 2, 1, 4>(st, one, tab, n, blocks);
    case 53: return go<16, 16, 3, 2, 2>(st, one, tab, n, blocks);
    default: set_error("no such tile sweep"); return BLZ_E_INVALID;
    }
}

// How `sweeps` sweeps are cut into launches: an even number of them (home
// planes -> spare -> home), as few as a family's longest launch allows, of
// nearly equal lengths of two sweeps at least. Of four sweeps or more that
// leaves at most one over (of 7, with three sweeps a launch), for the caller.
struct Plan {
    int launches = 0, shortest = 0, longer = 0, left = 0; // `longer` launches have shortest + 1 sweeps
};
Plan cut_into(int sweeps, int tmax) {
    Plan p;
    p.launches = 2 * ((sweeps + 2 * tmax - 1) / (2 * tmax));
    if (sweeps < 2 * p.launches) p.launches -= 2;
    const int n = std::min(sweeps, p.launches * tmax);
    p.left = sweeps - n;
    if (p.launches) {
        p.shortest = n / p.launches;
        p.longer = n % p.launches;
    }
    return p;
}
Plan plan_of(int family, int sweeps) {
    const int tmax = kFamilies[family].tmax;
    if (kFamilies[family].usual == 2) { // launches of two, a few of three for what is left
        Plan p;
        p.launches = sweeps / 4 * 2;
        p.shortest = 2;
        p.longer = std::min(sweeps - 2 * p.launches, p.launches);
        p.left = sweeps - 2 * p.launches - p.longer;
        return p;
    }
    const Plan p = cut_into(sweeps, tmax);
    if (tmax < 5) return p;
    // five sweeps in a launch need two items per wave: taken where they save
    // more launches than they cost (us per launch of 2 .. 5 sweeps at 32^3:
    // 10 sweeps are 2 x 5 in 29 us against 3 + 3 + 2 + 2 in 32, 100 sweeps
    // 26 launches of 4 and 3 in 259 us against 20 of 5 in 286)
    constexpr double us[] = {0.0, 0.0, 7.2, 8.6, 10.2, 14.3, 14.3};
    auto cost = [&](const Plan& q) {
        return (q.launches - q.longer) * us[q.shortest] + q.longer * us[q.shortest + 1] + 10.0 * q.left;
    };
    const Plan q = cut_into(sweeps, kFamilies[family].usual);
    return cost(q) <= cost(p) ? q : p;
}

} // namespace

// The tile for a W x H slab: the smallest of which every CU (256) gets at most
// one; a smaller tile has more rim to compute again and takes turns, a larger
// one leaves CUs idle. us per sweep on random pressure, calls of 120 sweeps, of
// 4x4 / 8x4 / 8x8 / 16x16 tiles: 64^3 3.8 / 4.1 / 4.5 / 7.3, 90x75x62 5.3 / 4.3 /
// 4.8 / 7.4, 128^3 15.3 / 8.0 / 7.1 / 11.8; of 8x8 / 16x8 / 16x12 / 16x16: 144^3
// 14.2 / 10.0 / 11.2 / 13.0, 160^3 15.5 / 10.8 / 12.0 / 14.1, 192^3 26.1 / 16.9 /
// 13.9 / 16.3, 256x128x256 22.4 / 15.5 / 17.4 / 20.4; of the last three: 224^3
// 20.4 / 25.1 / 18.8, 256^3 25.3 / 29.4 / 22.9.
int tile_family(int W, int H) {
    for (int f = 0; f < TILE_FAMILIES - 1; ++f)
        if (tile_count(f, W, H) <= 256) return f;
    return TILE_FAMILIES - 1;
}

int tile_count(int family, int W, int H) {
    const Family& f = kFamilies[family];
    return ((W + f.bx - 1) / f.bx) * ((H + f.by - 1) / f.by);
}

// `sweeps` (four or more) less *left of them, alternately as a and as b say: the two
// directions of one grid (na = 0) or of a table of na grids
int launch_tile_sweeps(hipStream_t st, int family, const FusedScene* a, const FusedScene* b, int na, int blocks,
                       int sweeps, int* launches, int* left) {
    const Plan p = plan_of(family, sweeps);
    for (int l = 0; l < p.launches; ++l) {
        const FusedScene* e = (l & 1) ? b : a;
        const int t = p.shortest + (l < p.longer ? 1 : 0);
        if (int rc = tile_sweeps(st, family, t, na ? nullptr : e, e, na, blocks)) return rc;
    }
    *launches = p.launches;
    *left = p.left;
    return BLZ_OK;
}

} // namespace blz
