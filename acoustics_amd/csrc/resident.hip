// resident.hip -- a block of steps of whole scenes held on the chip.
//
// Bound: the exchange between workgroups.  A step needs the neighbours' face
// pressures of the step before, and one hop through the memory side (a store
// of one workgroup to a load of another) takes 1.3-1.6 us with up to 256
// workgroups in flight, 1.9 us with 512, 3.0 us with 1024 (a bare exchange of
// 1024 words each); nothing else is read from or written to memory.  Measured
// per step: 64^3 with a 10-cell PML (206 workgroups) 2.1 us, of which the
// arithmetic alone 0.9 and the exchange alone 1.5 (the step kernels: 6.0);
// 128^3 with a 12-cell PML (733) 5.2 us, 2.9 and 5.0 (12.3).
//
// * Each face pressure travels in one 8-byte word with the step's tag above
//   it, so the data is its own flag: no store is waited for before a flag is
//   raised, and no load follows a flag (with flags and 4-byte data the bare
//   exchange took 1.8-2.4 us with 256 workgroups, 3.1-4.0 with 1024).
// * The words of a face are contiguous over lanes and start on a 128-byte
//   line (128^3: 6.4 -> 5.9 us per step; word by column instead of by lane, a
//   bare exchange took 14-24 us).
// * No lane branches on whether it has a word, and what only some steps or
//   tiles need (scene pointers for sources, records, rarer listener terms) is
//   loaded where it is used: 64^3 2.95 -> 2.39 us per step.
// * Cells' PML and leapfrog history is in registers, pressures in two LDS
//   buffers with x fastest, so a thread's column and its four neighbours'
//   columns are 16-byte reads.
#include <climits>

#include <hip/hip_ext.h>

#include "resident.h"
#include "stencil.h"

namespace fdtd {

namespace {

template <int SHAPE>
struct Shape;
// small grids: as many workgroups as possible
template <>
struct Shape<RES_FINE> {
    static constexpr int plain = 8, one = 8, more = 8, cs = 12, words = 4, recs = 2, waves = 3, lds = 4608;
    static constexpr bool in_place = false;
};
// larger grids: as many cells per workgroup as registers and LDS hold
template <>
struct Shape<RES_COARSE> {
    static constexpr int plain = 16, one = 12, more = 8, cs = 20, words = 6, recs = 3, waves = 3, lds = 6500;
    static constexpr bool in_place = false;
};
// grids beyond that: two workgroups a compute unit with 256 registers a lane,
// and pressures in one LDS buffer, so new ones wait in registers for a barrier.
// Slower where RES_COARSE fits (128^3 8.4 us per step against 5.3: two waves a
// SIMD hide less), faster than the step kernels beyond (144x146x144 7.9 us against 14.6).
template <>
struct Shape<RES_LARGE> {
    static constexpr int plain = 32, one = 24, more = 16, cs = 36, words = 10, recs = 3, waves = 2, lds = 15000;
    static constexpr bool in_place = true;
};

typedef unsigned long long u64;

__device__ __forceinline__ void send_word(AS_GLOBAL u64 *p, u64 v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 take_word(const AS_GLOBAL u64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The value, computed anew: offsets of the last stores would otherwise be
// carried in registers through all steps.
__device__ __forceinline__ int anew(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// face word w of a tile: the face, and the cell of that face (LDS place of
// the cell itself and of its neighbour across the face, global cell across it)
struct FaceCell {
    int own, halo;      // LDS words
    int i, j, k;        // the neighbour's cell (tile's frame)
    bool real;          // (the last words of a face stand for no cell)
};

// Words of a face, rounded up to whole 128-byte lines: a line then has one
// sender per neighbour.
__device__ __forceinline__ int face_words(int n) { return (n + 15) & ~15; }

// a[d] of a struct in device memory (a copy of it that is indexed by a variable
// would go to scratch memory)
template <class T>
__device__ __forceinline__ T pick(const T (&a)[3], int d) { return cmem(&a[0])[d]; }

// a tile's axes in the grid: its columns', and the one across
__device__ __forceinline__ int column_axis(const ResTile &t) { return t.swap ? 1 : 0; }
__device__ __forceinline__ int across_axis(const ResTile &t) { return t.swap ? 0 : 1; }
__device__ __forceinline__ int column_stride(const SceneDev &S, const ResTile &t) { return t.swap ? S.sy : S.sx; }
__device__ __forceinline__ int across_stride(const SceneDev &S, const ResTile &t) { return t.swap ? S.sx : S.sy; }

template <int CS>
__device__ __forceinline__ FaceCell face_cell(const ResTile &t, int w)
{
    const int nyz = face_words(t.by * t.bz), nxz = face_words(t.bx * t.bz), nxy = face_words(t.bx * t.by);
    const int P = t.pitch;
    FaceCell f;
    if (w < 2 * nyz) {
        const int hi = w >= nyz, c = w - hi * nyz, y = c / t.bz, z = c - y * t.bz;
        const int col = (y + 1) * P + (z + 1) * CS;
        f.own = col + (hi ? t.bx - 1 : 0);
        f.halo = col + (hi ? t.bx : CS - 1);
        f.i = hi ? t.i0 + t.bx : t.i0 - 1;
        f.j = t.j0 + y;
        f.k = t.k0 + z;
        f.real = y < t.by;
        return f;
    }
    w -= 2 * nyz;
    if (w < 2 * nxz) {
        const int hi = w >= nxz, c = w - hi * nxz, x = c / t.bz, z = c - x * t.bz;
        f.own = (hi ? t.by : 1) * P + (z + 1) * CS + x;
        f.halo = (hi ? t.by + 1 : 0) * P + (z + 1) * CS + x;
        f.i = t.i0 + x;
        f.j = hi ? t.j0 + t.by : t.j0 - 1;
        f.k = t.k0 + z;
        f.real = x < t.bx;
        return f;
    }
    w -= 2 * nxz;
    const int hi = w >= nxy, c = w - hi * nxy, x = c / t.by, y = c - x * t.by;
    f.own = (y + 1) * P + (hi ? t.bz : 1) * CS + x;
    f.halo = (y + 1) * P + (hi ? t.bz + 1 : 0) * CS + x;
    f.i = t.i0 + x;
    f.j = t.j0 + y;
    f.k = hi ? t.k0 + t.bz : t.k0 - 1;
    f.real = x < t.bx;
    return f;
}

// Fills a scene's route table, one workgroup per tile: the tile on the other
// side of each face word and the word there that stands for the own cell.  A
// wall's words go to the tile itself (the halo beyond a wall equals the cell
// before it; the wall face's zero factors keep its velocity at zero), and lanes
// without a word share one more that goes nowhere else: every lane of the
// exchange then does the same.
template <int CS>
__global__ __launch_bounds__(RES_THREADS) void route_kernel(const ResScene *__restrict__ scene)
{
    const ResScene R = *cmem(scene);
    const SceneDev S = *cmem(R.S);
    const ResTile t = cmem(R.tiles)[blockIdx.x];
    for (int w = (int)threadIdx.x; w <= t.words; w += RES_THREADS) {
        ResRoute r;
        r.to = t.word0 + (uint32_t)w;
        r.lds = 0;              // (an unused corner of the halo)
        FaceCell f;
        f.real = false;
        if (w < t.words) f = face_cell<CS>(t, w);
        if (!f.real) {
            gmem(R.route)[t.word0 + (uint32_t)w] = r;
            continue;
        }
        r.lds = (uint32_t)f.own | ((uint32_t)f.halo << 16);
        const int x[3] = {t.swap ? f.j : f.i, t.swap ? f.i : f.j, f.k};
        if (x[0] >= 0 && x[1] >= 0 && x[2] >= 0 && x[0] < S.n[0] && x[1] < S.n[1] && x[2] < S.n[2]) {
            // the face's axis, and whether it is the tile's low one
            const int a = f.i < t.i0 || f.i >= t.i0 + t.bx ? column_axis(t) : f.j < t.j0 || f.j >= t.j0 + t.by ? across_axis(t) : 2;
            const bool low = f.i < t.i0 || f.j < t.j0 || f.k < t.k0;
            for (int b = 0; b < R.nboxes; ++b) {
                const ResBox B = cmem(R.boxes)[b];
                int at[3];
                bool in = true;
                for (int d = 0; d < 3; ++d) {
                    at[d] = x[d] - B.lo[d];
                    in = in && at[d] >= 0 && at[d] < B.len[d];
                }
                if (!in) continue;
                const int q = B.first + ((at[0] / B.size[0]) * B.count[1] + at[1] / B.size[1]) * B.count[2] + at[2] / B.size[2];
                const ResTile o = gmem(R.tiles)[q];
                const int nyz = face_words(o.by * o.bz), nxz = face_words(o.bx * o.bz), nxy = face_words(o.bx * o.by);
                const int li = (o.swap ? x[1] : x[0]) - o.i0, lj = (o.swap ? x[0] : x[1]) - o.j0, lk = x[2] - o.k0;
                // the own cell is across the neighbour's opposite face
                int word;
                if (a == column_axis(o)) word = (low ? nyz : 0) + lj * o.bz + lk;
                else if (a == across_axis(o)) word = 2 * nyz + (low ? nxz : 0) + li * o.bz + lk;
                else word = 2 * (nyz + nxz) + (low ? nxy : 0) + li * o.by + lj;
                r.to = o.word0 + (uint32_t)word;
                break;
            }
        }
        gmem(R.route)[t.word0 + (uint32_t)w] = r;
    }
}

// the table entry of face / cell i along axis d: a wall face gets zero factors
__device__ __forceinline__ float4 table_entry(const SceneDev *S, int d, int i)
{
    float4 c = gmem(pick(S->coef, d))[min(i, pick(S->n, d))];
    if (i <= 0 || i >= pick(S->n, d)) { c.x = 0.f; c.y = 0.f; }
    return c;
}

// The pointer, read anew: what is loaded through it is loaded there, and not
// carried in scalar registers through all steps.
template <class T>
__device__ __forceinline__ const T *anew(const T *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

template <class T>
__device__ __forceinline__ AS_GLOBAL T *at_byte(T *base, uint32_t off)
{
    return (AS_GLOBAL T *)((AS_GLOBAL char *)base + off);
}

// What a workgroup carries through its steps besides the class's registers.
template <int SHAPE>
struct Frame {
    using C = Shape<SHAPE>;
    const SceneDev *scene;
    const ResScene *res;
    const ResTile *tile;
    float *A, *B;               // this step's pressures and the next's, in LDS
    float4 *X;                  // table of the tile's cells and faces along its columns, in LDS
    long long step0;
    int steps;
    uint32_t tag;
    int *trouble;
    int bx;
    // own column
    bool act;
    int ly, lz, col;            // col: LDS word of the column's first cell
    int P;                      // LDS words from a column to the next along y
    // face words: where they go (bytes), LDS places of the own cell and of the halo (bytes, 16 bits each)
    u64 *words;
    uint32_t half;              // bytes of one parity's words
    uint32_t to[C::words], lds[C::words];
    uint32_t word0;             // byte of this tile's first word
    int nwords;
    // the tile's listener terms: this thread's first one
    bool terms_here, has_term, more_terms;
    double *term_to;            // its place in ring row 0
    double term_beta;
    int term_at;
    int ring0, cap;             // ring row of step0, rows
    uint32_t row_bytes;
    bool stuck;
    // amplitude of the first pressure source in the step to come, fetched
    // while the exchange of the step before runs; sources (0: none reaches the tile)
    int src, amp_last;
    const AS_GLOBAL float *src_tab;
    float amp;

    // the scene, for code off the step loop's usual path
    __device__ __forceinline__ SceneDev scene_now() const { return *cmem(anew(scene)); }

    __device__ __forceinline__ static int place(const SceneDev &S, const ResTile &t, int cell)
    {
        const int i = cell / S.sx, r = cell - i * S.sx, j = r / S.sy, k = r - j * S.sy;
        const int u = t.swap ? j : i, v = t.swap ? i : j;
        return (v - t.j0 + 1) * t.pitch + (k - t.k0 + 1) * C::cs + (u - t.i0);
    }

    // p^{step} of the tile and its halo, both buffers cleared before
    __device__ __forceinline__ void load(const SceneDev &S, const ResScene &R, const ResTile &t)
    {
        const int tid = (int)threadIdx.x, n = (C::in_place ? 1 : 2) * C::lds;
        for (int q = tid; q < n; q += RES_THREADS) A[q] = 0.f;
        bx = t.bx;
        P = t.pitch;
        act = tid < t.by * t.bz;
        ly = act ? tid / t.bz : 0;
        lz = act ? tid - ly * t.bz : 0;
        col = (ly + 1) * P + (lz + 1) * C::cs;
        if (tid <= C::plain) X[tid] = table_entry(scene, column_axis(t), t.i0 + tid);
        __syncthreads();
        const AS_GLOBAL float *pc = gmem(S.field + (size_t)slot_cur(step0) * S.npad);
        if (act) {
            const int su = column_stride(S, t), idx = t.i0 * su + (t.j0 + ly) * across_stride(S, t) + t.k0 + lz;
#pragma unroll
            for (int i = 0; i < C::plain; ++i)
                if (i < t.bx) A[col + i] = pc[idx + i * su];
        }
        words = R.words;
        half = R.nwords * 8u;
        word0 = t.word0 * 8u;
        nwords = t.words;
#pragma unroll
        for (int m = 0; m < C::words; ++m) {
            const int w = min(tid + m * RES_THREADS, t.words);
            const ResRoute r = gmem(R.route)[t.word0 + (uint32_t)w];
            to[m] = r.to * 8u;
            lds[m] = r.lds * 4u;
            if (w < t.words) {
                const FaceCell f = face_cell<C::cs>(t, w);
                const int i = t.swap ? f.j : f.i, j = t.swap ? f.i : f.j;
                if (f.real && i >= 0 && j >= 0 && f.k >= 0 && i < S.n[0] && j < S.n[1] && f.k < S.n[2])
                    A[f.halo] = pc[i * S.sx + j * S.sy + f.k];
            }
        }
        // one term per thread of the usual kind (a cell's new pressure) is
        // kept ready; others are looked up each step
        terms_here = t.te > t.tb;
        has_term = t.tb + tid < t.te;
        term_at = 0;
        cap = S.cap;
        ring0 = (int)(step0 % S.cap);
        row_bytes = 8u * (uint32_t)S.T;
        more_terms = t.te - t.tb > RES_THREADS;
        if (has_term) {
            const TermRef r = gmem(R.terms)[t.tb + tid];
            term_to = S.terms + r.slot;
            term_beta = r.beta;
            if (r.kind == 0) term_at = place(S, t, r.cell);
            else { has_term = false; more_terms = true; }
        }
        more_terms = __any(more_terms);
        stuck = false;
        src = t.src ? S.n_psrc : 0;
        src_tab = gmem(S.src_tab);
        amp_last = S.amp_rows - 1;
        amp = 0.f;
        if (src) {
            const PSrcDev ps = cmem(S.psrc)[0];
            const int gu = t.swap ? ps.goff[1] : ps.goff[0], n = t.swap ? S.n[1] : S.n[0];
            if (tid < C::plain) along()[tid] = gmem(S.gtab)[gu + min(t.i0 + tid, n - 1)];
        }
        fetch_amp(step0);
    }

    __device__ __forceinline__ void fetch_amp(long long step)
    {
        if (src) amp = src_tab[(int)(step & amp_last) * src];
    }
    // (an amplitude of zero, once the pulse is over, adds nothing)
    __device__ __forceinline__ bool sounding() const { return src && (amp != 0.f || src > 1); }
    // the first source's factor along the columns (after the table in LDS) ...
    __device__ __forceinline__ float *along() const { return (float *)(X + C::plain + 1); }
    // ... and across them and along z, for a step's add_sources
    struct Across { float v, z; };
    __device__ __forceinline__ Across across(const SceneDev &Z, const ResTile &u) const
    {
        const PSrcDev ps = cmem(Z.psrc)[0];
        const AS_GLOBAL float *g = gmem(Z.gtab);
        return {g[(u.swap ? ps.goff[0] : ps.goff[1]) + u.j0 + ly], g[ps.goff[2] + u.k0 + lz]};
    }
    // the pressure sources' S dt at cell i of the own column in step `step`, added to v.
    // The first one's factors are at hand: a staggered pulse never ends, and
    // loaded cell by cell they held up its tiles in every step (150x97x133:
    // 10.7 us per step, now 7.0; kept in registers for all steps they cost the
    // other tiles 3%)
    __device__ __forceinline__ float add_sources(const SceneDev &Z, const ResTile &u, Across w, long long step, int i, float v) const
    {
        // (only the in-place shape's tiles swap)
        if (amp != 0.f) v = C::in_place && u.swap ? add_source(v, amp, w.v, along()[i], w.z) : add_source(v, amp, along()[i], w.v, w.z);
        for (int p = 1; p < Z.n_psrc; ++p) {
            const float a = gmem(Z.src_tab)[amp_row(Z, step) * Z.n_psrc + p];
            if (a == 0.f) continue;
            const PSrcDev ps = cmem(Z.psrc)[p];
            const AS_GLOBAL float *g = gmem(Z.gtab);
            const int x = u.swap ? u.j0 + ly : min(u.i0 + i, Z.n[0] - 1), y = u.swap ? min(u.i0 + i, Z.n[1] - 1) : u.j0 + ly;
            v = add_source(v, a, g[ps.goff[0] + x], g[ps.goff[1] + y], g[ps.goff[2] + u.k0 + lz]);
        }
        return v;
    }

    // Step s has been made: a cell's term takes its new pressure (in B), a
    // ghost's its value in that step (from A; in place, before the cells are
    // written, with GHOSTS).
    template <bool GHOSTS = false>
    __device__ __forceinline__ void terms(int s) const
    {
        if (!terms_here) return;
        const int row = ring0 + s < cap ? ring0 + s : ring0 + s - cap;
        if (has_term && !GHOSTS) *(AS_GLOBAL double *)((AS_GLOBAL char *)term_to + (size_t)row * row_bytes) = term_beta * (double)B[term_at];
        if (!more_terms) return;
        const SceneDev S = scene_now();
        const ResScene R = *cmem(anew(res));
        const ResTile t = *cmem(anew(tile));
        for (int q = t.tb + (int)threadIdx.x; q < t.te; q += RES_THREADS) {
            const TermRef r = gmem(R.terms)[q];
            if (r.kind == 0 && (GHOSTS || q < t.tb + RES_THREADS)) continue;
            if (C::in_place && r.kind != 0 && !GHOSTS) continue;
            double v;
            if (r.kind == 0) v = (double)B[place(S, t, r.cell)];
            else {
                const GhostDev g = gmem(S.ghosts)[r.cell];
                v = (double)A[place(S, t, g.nbr)] + raster_accel_term(S, g, step0 + s);
            }
            gmem(S.terms)[(size_t)row * S.T + r.slot] = r.beta * v;
        }
    }

    // sends the tile's faces of step s, just made (all of B's own cells are
    // written and visible)
    __device__ __forceinline__ void send(int s) const
    {
        const uint32_t mark = tag + (uint32_t)s;
        u64 *buf = words + ((mark & 1u) ? half / 8u : 0u);
        float v[C::words];
#pragma unroll
        for (int m = 0; m < C::words; ++m) v[m] = *(const float *)((const char *)B + (lds[m] & 0xffffu));
#pragma unroll
        for (int m = 0; m < C::words; ++m) send_word(at_byte(buf, to[m]), ((u64)mark << 32) | __float_as_uint(v[m]));
    }
    // waits for the neighbours' faces of step s
    __device__ __forceinline__ void receive(int s)
    {
        const uint32_t mark = tag + (uint32_t)s;
        u64 *buf = words + ((mark & 1u) ? half / 8u : 0u);
        u64 v[C::words];
        for (int spins = 0;; ++spins) {
            uint32_t miss = 0;
#pragma unroll
            for (int m = 0; m < C::words; ++m)
                v[m] = take_word(at_byte(buf, word0 + 8u * (uint32_t)min((int)threadIdx.x + m * RES_THREADS, nwords)));
#pragma unroll
            for (int m = 0; m < C::words; ++m) miss |= (uint32_t)(v[m] >> 32) ^ mark;
            if (miss == 0 || stuck) break;
            if (spins > (1 << 22)) {
                // the neighbours are on the device, so this does not happen;
                // it keeps every wave's exit certain
                stuck = true;
                __hip_atomic_store(const_cast<int *>(anew((const int *)trouble)), 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
#pragma unroll
        for (int m = 0; m < C::words; ++m) *(float *)((char *)B + (lds[m] >> 16)) = __uint_as_float((uint32_t)v[m]);
    }
    __device__ __forceinline__ void turn()
    {
        float *q = A;
        A = B;
        B = q;
    }

    // (in place, the last step) the level before the newest, which the step overwrites
    __device__ __forceinline__ void store_old() const
    {
        if (!act) return;
        const SceneDev S = scene_now();
        const ResTile t = *cmem(anew(tile));
        AS_GLOBAL float *pp = gmem(S.field + (size_t)slot_next(step0 + steps) * S.npad);
        const int su = column_stride(S, t), idx = t.i0 * su + (t.j0 + anew(ly)) * across_stride(S, t) + t.k0 + lz;
        for (int i = 0; i < t.bx; ++i) pp[idx + i * su] = A[col + i];
    }

    // the last two levels of the own cells, into the slots of step step0 + steps
    __device__ __forceinline__ void store_pressure(const SceneDev &S, const ResTile &t) const
    {
        if (!act) return;
        const long long s = step0 + steps;
        AS_GLOBAL float *pc = gmem(S.field + (size_t)slot_cur(s) * S.npad), *pp = gmem(S.field + (size_t)slot_next(s) * S.npad);
        const int su = column_stride(S, t), idx = t.i0 * su + (t.j0 + anew(ly)) * across_stride(S, t) + t.k0 + lz;
#pragma unroll
        for (int i = 0; i < C::plain; ++i)
            if (i < t.bx) {
                pc[idx + i * su] = A[col + i];
                if (!C::in_place) pp[idx + i * su] = B[col + i];
            }
    }
};

// The own column, the x halos beside it, and four cells of the columns around
// it: cells 4 q .. 4 q + 3.
template <int CS, int NB>
struct Column {
    float c[NB + 1], before;    // cells 0 .. NB (cell bx is the x-high halo); the x-low halo
    __device__ __forceinline__ void load(const float *A, int col)
    {
#pragma unroll
        for (int q = 0; q < NB / 4; ++q) {
            const float4 v = *(const float4 *)(A + col + 4 * q);
            c[4 * q] = v.x; c[4 * q + 1] = v.y; c[4 * q + 2] = v.z; c[4 * q + 3] = v.w;
        }
        c[NB] = A[col + NB];
        before = A[col + CS - 1];
    }
};
struct Quad {
    float yl[4], yr[4], zl[4], zr[4];
};
template <int CS>
__device__ __forceinline__ Quad quad(const float *A, int col, int P, int q)
{
    Quad u;
    const float *a = A + col + 4 * q;
    const float4 yl = *(const float4 *)(a - P), yr = *(const float4 *)(a + P);
    const float4 zl = *(const float4 *)(a - CS), zr = *(const float4 *)(a + CS);
    u.yl[0] = yl.x; u.yl[1] = yl.y; u.yl[2] = yl.z; u.yl[3] = yl.w;
    u.yr[0] = yr.x; u.yr[1] = yr.y; u.yr[2] = yr.z; u.yr[3] = yr.w;
    u.zl[0] = zl.x; u.zl[1] = zl.y; u.zl[2] = zl.z; u.zl[3] = zl.w;
    u.zr[0] = zr.x; u.zr[1] = zr.y; u.zr[2] = zr.z; u.zr[3] = zr.w;
    return u;
}
// Writes cells 4 q .. 4 q + 3 of the column.  Cells past the tile's last are
// written too: the first of them is the place of the x-high halo, which the
// exchange then fills in, and no cell of the tile reads the others.
__device__ __forceinline__ void put_quad(float *B, int col, int q, const float *o)
{
    *(float4 *)(B + col + 4 * q) = make_float4(o[0], o[1], o[2], o[3]);
}

// In place: every thread has read what it needs of this step's pressures, and
// may write the next ones.
template <int SHAPE>
__device__ __forceinline__ void before_writes(Frame<SHAPE> &F, int s)
{
    if constexpr (Shape<SHAPE>::in_place) {
        F.template terms<true>(s);
        if (s == F.steps - 1) F.store_old();
        __syncthreads();
    }
}
// Writes a column of new pressures; (in place) cells past the tile's last as put_quad.
template <int NB>
__device__ __forceinline__ void put_column(float *B, int col, int bx, const float *o)
{
#pragma unroll
    for (int q = 0; q < NB / 4; ++q)
        if (4 * q < bx) put_quad(B, col, q, o + 4 * q);
}

// Undamped cells: leapfrog, pressure sources, and the object-adjacent cells
// of the tile in FP64 by one thread per record.
// INC: the merged staggered scheme, which keeps the increment in place of the
// last level.
template <int SHAPE, bool INC>
__device__ __forceinline__ void run_plain(Frame<SHAPE> &F, const SceneDev &S, const ResTile &t)
{
    using C = Shape<SHAPE>;
    constexpr int NB = C::plain, NR = C::recs;
    const int tid = (int)threadIdx.x;
    float prev[NB];
    uint32_t skip = 0;
    const float lam2 = S.lam2f;
    const bool skips = t.skip, records = t.re > t.rb;
    const int j = t.j0 + F.ly, k = t.k0 + F.lz;   // (threads without a column: the first one's)
    {
        const AS_GLOBAL float *pp = INC ? gmem(S.inc) : gmem(S.field + (size_t)slot_next(F.step0) * S.npad);
        const int idx = t.i0 * S.sx + j * S.sy + k;
#pragma unroll
        for (int i = 0; i < NB; ++i) prev[i] = pp[idx + min(i, t.bx - 1) * S.sx];
        if (t.skip)
            for (int i = 0; i < t.bx; ++i) skip |= (gmem(S.skip)[idx + i * S.sx] ? 1u : 0u) << i;
    }
    // records: place, last level, the ghost term's factor per side
    int rat[NR], rmask[NR], robj[NR];
    float rprev[NR];
    double rk[NR][6];
    if (t.re > t.rb) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            rat[r] = -1;
            const int q = t.rb + tid + r * RES_THREADS;
            if (q >= t.re) continue;
            const SpecialRec rec = gmem(S.recs)[gmem(cmem(F.res)->recs)[q]];
            rat[r] = F.place(S, t, rec.cell);
            rprev[r] = gmem(S.field + (size_t)slot_next(F.step0) * S.npad)[rec.cell];
            rmask[r] = (rec.flags & 1) << 6 | rat[r] % F.P % C::cs << 8;   // (its x place above the bits)
            robj[r] = 0;
            for (int e = 0; e < 6; ++e) {
                rk[r][e] = 0.0;
                if (rec.gid[e] < 0) continue;
                const GhostDev gd = gmem(S.ghosts)[rec.gid[e]];
                rmask[r] |= 1 << e;
                robj[r] = gd.obj;
                rk[r][e] = gd.k_raster;
            }
        }
    }
    // accelerations of a step, fetched while the exchange of the one before runs
    double racc[NR];
    auto accelerations = [&](long long step) {
        if (!records) return;
        const SceneDev Z = F.scene_now();
#pragma unroll
        for (int r = 0; r < NR; ++r) racc[r] = rat[r] >= 0 ? gmem(Z.acc_tab)[amp_row(Z, step) * Z.n_ch + robj[r]] : 0.0;
    };
    accelerations(F.step0);
    for (int s = 0; s < F.steps; ++s) {
        const long long step = F.step0 + s;
        // new pressures: four at a time, or (in place) in the column, from which
        // each cell has been read by the time it is replaced
        Column<C::cs, NB> w;
        if (F.act) {
            w.load(F.A, F.col);
            float left = w.before;
#pragma unroll
            for (int q = 0; q < NB / 4; ++q) {
                if (4 * q >= F.bx) continue;
                const Quad u = quad<C::cs>(F.A, F.col, F.P, q);
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * q + e;
                    const float c = w.c[i], xm = C::in_place ? left : i ? w.c[i - 1] : w.before, xp = w.c[i + 1];
                    if (INC) {
                        prev[i] = increment1(c, prev[i], xm, xp, u.yl[e], u.yr[e], u.zl[e], u.zr[e], lam2);
                        o[e] = c + prev[i];
                    } else {
                        o[e] = leapfrog1(c, prev[i], xm, xp, u.yl[e], u.yr[e], u.zl[e], u.zr[e], lam2);
                        prev[i] = c;
                    }
                    if (C::in_place) { left = c; w.c[i] = o[e]; }
                }
                if constexpr (!C::in_place) {
                    if (!skips) put_quad(F.B, F.col, q, o);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (4 * q + e < F.bx && !(skip >> (4 * q + e) & 1)) F.B[F.col + 4 * q + e] = o[e];
                    }
                }
            }
        }
        float rnow[NR];
        if (records) {
            const SceneDev Z = F.scene_now();
            const ResTile u = *cmem(anew(F.tile));
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                if (rat[r] < 0) continue;
                const float *a = F.A + rat[r];
                const int x = rmask[r] >> 8;
                const float cf = a[0];
                const double c = cf;
                const double nb[6] = {x == 0 ? a[C::cs - 1] : a[-1], a[1], a[-F.P], a[F.P], a[-C::cs], a[C::cs]};
                double g[6];
#pragma unroll
                for (int e = 0; e < 6; ++e) g[e] = (rmask[r] >> e & 1) ? c + rk[r][e] * racc[r] : 0.0;
                double lap = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    lap += ghost_lap_axis(Z.seven, rmask[r] >> (2 * d) & 1, rmask[r] >> (2 * d + 1) & 1, g[2 * d], g[2 * d + 1],
                                          nb[2 * d], nb[2 * d + 1], c);
                double pn = (rmask[r] >> 6 & 1) ? c : special_update(c, (double)rprev[r], lap, Z.lam2);
                if (Z.n_psrc > 0) {
                    const int y = rat[r] / F.P - 1, z = rat[r] % F.P / C::cs - 1;
                    for (int p = 0; p < Z.n_psrc; ++p) {
                        const PSrcDev ps = cmem(Z.psrc)[p];
                        const AS_GLOBAL float *g3 = gmem(Z.gtab);
                        pn += (double)(gmem(Z.src_tab)[amp_row(Z, step) * Z.n_psrc + p] * g3[ps.goff[0] + u.i0 + x] *
                                       g3[ps.goff[1] + u.j0 + y] * g3[ps.goff[2] + u.k0 + z]);
                    }
                }
                rprev[r] = cf;
                rnow[r] = (float)pn;
            }
        }
        before_writes(F, s);
        if (F.act) {
            if constexpr (C::in_place) {
                if (!skips) put_column<NB>(F.B, F.col, F.bx, w.c);
                else {
#pragma unroll
                    for (int i = 0; i < NB; ++i)
                        if (i < F.bx && !(skip >> i & 1)) F.B[F.col + i] = w.c[i];
                }
            }
            if (F.sounding()) {
                const SceneDev Z = F.scene_now();
                const ResTile u = *cmem(anew(F.tile));
                const auto w = F.across(Z, u);
                for (int i = 0; i < F.bx; ++i)
                    if (!(skip >> i & 1)) {
                        float &o = F.B[F.col + i];
                        o = INC ? fmaf(3.f, F.add_sources(Z, u, w, step, i, 0.f), o) : F.add_sources(Z, u, w, step, i, o);
                    }
            }
        }
        if (records) {
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (rat[r] >= 0) F.B[rat[r]] = rnow[r];
        }
        __syncthreads();
        F.send(s);
        F.terms(s);
        F.fetch_amp(step + 1);
        accelerations(step + 1);
        F.receive(s);
        F.turn();
        __syncthreads();
    }
    const SceneDev Z = F.scene_now();
    const ResTile u = *cmem(anew(F.tile));
    F.store_pressure(Z, u);
    if (!INC || !F.act) return;
    const int idx = u.i0 * Z.sx + (u.j0 + anew(F.ly)) * Z.sy + u.k0 + F.lz;
#pragma unroll
    for (int i = 0; i < NB; ++i)
        if (i < u.bx) gmem(Z.inc)[idx + i * Z.sx] = prev[i];
}

// Face and cell coefficients of the own column along y or z.
struct AxisCoef {
    float l1, l2, r1, r2, c3, c5;   // faces low and high {f1, f2}, cell {f3, f5/h}; a wall face stays at zero
};
__device__ __forceinline__ AxisCoef axis_coef(const SceneDev *S, int d, int i)
{
    const float4 lo = gmem(pick(S->coef, d))[i], hi = gmem(pick(S->coef, d))[i + 1];
    AxisCoef a;
    a.l1 = i > 0 ? lo.x : 0.f;
    a.l2 = i > 0 ? lo.y : 0.f;
    a.r1 = i + 1 < pick(S->n, d) ? hi.x : 0.f;
    a.r2 = i + 1 < pick(S->n, d) ? hi.y : 0.f;
    a.c3 = lo.z;
    a.c5 = lo.w;
    return a;
}
__device__ __forceinline__ float face_step(float f1, float f2, float v, float pl, float pr)
{
    return fmaf(f2, pr - pl, f1 * v);
}
__device__ __forceinline__ float split_step(float f3, float f5, float q, float dv)
{
    return fmaf(f5, dv, f3 * q);
}
// compact offsets of the own column's cells and faces in its slab: the cell's,
// and the low faces' along the tile's axes, of column cell i
struct SlabAt {
    int c, cu, u, uu, v, vu, vh, w, wu;
    __device__ SlabAt(const PmlSlab &s, const ResTile &t, int ly, int lz)
    {
        const int e1 = s.e[1], e2 = s.e[2];
        const int x = (t.swap ? t.j0 + ly : t.i0) - s.lo[0], y = (t.swap ? t.i0 : t.j0 + ly) - s.lo[1], z = t.k0 + lz - s.lo[2];
        c = (x * e1 + y) * e2 + z;                   // and the x face
        const int yf = (x * (e1 + 1) + y) * e2 + z;  // the y face
        w = (x * e1 + y) * (e2 + 1) + z;
        cu = t.swap ? e2 : e1 * e2;
        u = t.swap ? yf : c;
        uu = cu;
        v = t.swap ? c : yf;
        vu = t.swap ? e2 : (e1 + 1) * e2;
        vh = t.swap ? e1 * e2 : e2;
        wu = t.swap ? e2 + 1 : e1 * (e2 + 1);
    }
    __device__ __forceinline__ int cell(int i) const { return c + i * cu; }
    __device__ __forceinline__ int fu(int i) const { return u + i * uu; }
    __device__ __forceinline__ int fv(int i, int h) const { return v + i * vu + h * vh; }
    __device__ __forceinline__ int fw(int i, int h) const { return w + i * wu + h; }
};

// Cells damped along axis D of the tile only (the merged PML state): pDir along
// it, both faces along it, and the increment of the transverse sum.
template <int SHAPE, int D>
__device__ __forceinline__ void run_one(Frame<SHAPE> &F, const SceneDev &S, const ResTile &t)
{
    using C = Shape<SHAPE>;
    constexpr int NB = C::one;
    const PmlSlab sl = cmem(S.slabs)[t.slab];
    const SlabAt at(sl, t, F.ly, F.lz);
    const int gu = column_axis(t), gv = across_axis(t), g = D == 0 ? gu : D == 1 ? gv : 2;   // axes of the grid; g the damped one
    AS_GLOBAL float *pq = gmem(pick(F.scene->pd, g) + sl.cell_base), *pi = gmem(pick(F.scene->pd, g == 0 ? 1 : 0) + sl.cell_base);
    float q0[NB], dd[NB], vl[D == 0 ? NB + 1 : NB], vr[D == 0 ? 1 : NB];
    const AxisCoef cy = axis_coef(F.scene, gv, t.j0 + F.ly), cz = axis_coef(F.scene, 2, t.k0 + F.lz);
    {
        const AS_GLOBAL float *v = gmem((F.step0 & 1 ? pick(F.scene->vel[1], g) : pick(F.scene->vel[0], g)) + pick(S.slabs[t.slab].v_base, g));
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int e = min(i, t.bx - 1);
            q0[i] = pq[at.cell(e)];
            dd[i] = pi[at.cell(e)];
            if (D == 0) vl[i] = v[at.fu(e)];
            if (D == 1) { vl[i] = v[at.fv(e, 0)]; vr[i] = v[at.fv(e, 1)]; }
            if (D == 2) { vl[i] = v[at.fw(e, 0)]; vr[i] = v[at.fw(e, 1)]; }
        }
        if (D == 0) {
            // the high face of the last cell (compile-time places only)
            const float last = v[at.fu(t.bx)];
#pragma unroll
            for (int i = 1; i <= NB; ++i)
                if (i == t.bx) vl[i] = last;
        }
    }
    const float4 xp0 = cmem(pick(F.scene->coef, gu))[t.i0];   // D != 0: plain along the columns, one entry for all
    for (int s = 0; s < F.steps; ++s) {
        Column<C::cs, NB> w;
        if (F.act) {
            w.load(F.A, F.col);
            float left = w.before;
            float before = 0.f;                 // D == 0: the updated low face of the next cell
#pragma unroll
            for (int q = 0; q < NB / 4; ++q) {
                if (4 * q >= F.bx) continue;
                const Quad u = quad<C::cs>(F.A, F.col, F.P, q);
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * q + e;
                    const float c = w.c[i], xm = C::in_place ? left : i ? w.c[i - 1] : w.before, xp = w.c[i + 1];
                    float n, lap = 0.f;
                    const float qo = q0[i];
                    if (D == 0) {
                        const float4 xl = F.X[i], xr = F.X[i + 1];
                        if (i == 0) before = face_step(xl.x, xl.y, vl[0], xm, c);
                        const float after = face_step(xr.x, xr.y, vl[i + 1], c, xp);
                        n = split_step(xl.z, xl.w, qo, after - before);
                        vl[i] = before;
                        before = after;
                        if (e == 3) vl[i + 1] = after;
                    } else if (D == 1) {
                        vl[i] = face_step(cy.l1, cy.l2, vl[i], u.yl[e], c);
                        vr[i] = face_step(cy.r1, cy.r2, vr[i], c, u.yr[e]);
                        n = split_step(cy.c3, cy.c5, qo, vr[i] - vl[i]);
                    } else {
                        vl[i] = face_step(cz.l1, cz.l2, vl[i], u.zl[e], c);
                        vr[i] = face_step(cz.r1, cz.r2, vr[i], c, u.zr[e]);
                        n = split_step(cz.c3, cz.c5, qo, vr[i] - vl[i]);
                    }
                    if (D != 0) lap = transverse_add(lap, xp0.w, xp0.y, xp0.y, xm, c, xp);
                    if (D != 1) lap = transverse_add(lap, cy.c5, cy.l2, cy.r2, u.yl[e], c, u.yr[e]);
                    if (D != 2) lap = transverse_add(lap, cz.c5, cz.l2, cz.r2, u.zl[e], c, u.zr[e]);
                    const float dn = dd[i] + lap, dA = n - qo;
                    dd[i] = dn;
                    q0[i] = n;
                    o[e] = c + (dA + dn);
                    if (C::in_place) { left = c; w.c[i] = o[e]; }
                }
                if constexpr (!C::in_place) put_quad(F.B, F.col, q, o);
            }
        }
        before_writes(F, s);
        if constexpr (C::in_place) {
            if (F.act) put_column<NB>(F.B, F.col, F.bx, w.c);
        }
        if (F.act && F.sounding()) {
            // (staggered scheme) on both undamped axes
            const SceneDev Z = F.scene_now();
            const ResTile u = *cmem(anew(F.tile));
            const auto w = F.across(Z, u);
            for (int i = 0; i < F.bx; ++i) {
                float &o = F.B[F.col + i];
                o = fmaf(2.f, F.add_sources(Z, u, w, F.step0 + s, i, 0.f), o);
            }
        }
        __syncthreads();
        F.send(s);
        F.terms(s);
        F.fetch_amp(F.step0 + s + 1);
        F.receive(s);
        F.turn();
        __syncthreads();
    }
    const SceneDev Z = F.scene_now();
    const ResTile u = *cmem(anew(F.tile));
    F.store_pressure(Z, u);
    if (!F.act) return;
    const PmlSlab zl_ = cmem(Z.slabs)[u.slab];
    const SlabAt to(zl_, u, anew(F.ly), anew(F.lz));
    const int h = D == 0 ? column_axis(u) : D == 1 ? across_axis(u) : 2;
    AS_GLOBAL float *zq = gmem(pick(F.scene->pd, h) + zl_.cell_base), *zi = gmem(pick(F.scene->pd, h == 0 ? 1 : 0) + zl_.cell_base);
    AS_GLOBAL float *v = gmem(((F.step0 + F.steps) & 1 ? pick(F.scene->vel[1], h) : pick(F.scene->vel[0], h)) + pick(Z.slabs[u.slab].v_base, h));
#pragma unroll
    for (int i = 0; i <= NB; ++i) {
        if (i < NB && i < u.bx) {
            zq[to.cell(i)] = q0[i];
            zi[to.cell(i)] = dd[i];
            if (D == 1) { v[to.fv(i, 0)] = vl[i]; if (F.ly == u.by - 1) v[to.fv(i, 1)] = vr[i]; }
            if (D == 2) { v[to.fw(i, 0)] = vl[i]; if (F.lz == u.bz - 1) v[to.fw(i, 1)] = vr[i]; }
        }
        if (D == 0 && i <= u.bx) v[to.fu(i)] = vl[i];
    }
}

// Cells damped along two or three axes: three split pressures, the faces of
// all three axes (a face of two tiles is kept by both, computed alike).
template <int SHAPE>
__device__ __forceinline__ void run_more(Frame<SHAPE> &F, const SceneDev &S, const ResTile &t)
{
    using C = Shape<SHAPE>;
    constexpr int NB = C::more;
    const PmlSlab sl = cmem(S.slabs)[t.slab];
    const SlabAt at(sl, t, F.ly, F.lz);
    float q0[NB], q1[NB], q2[NB], vx[NB + 1], yl[NB], yr[NB], zl[NB], zr[NB];
    // (in the tile's frame)
    const int damped = t.swap ? (t.damped & 4) | (t.damped & 1) << 1 | (t.damped >> 1 & 1) : t.damped;
    const int gu = column_axis(t), gv = across_axis(t);
    const AxisCoef cy = axis_coef(F.scene, gv, t.j0 + F.ly), cz = axis_coef(F.scene, 2, t.k0 + F.lz);
    {
        const int b = (int)(F.step0 & 1);
        const AS_GLOBAL float *v0 = gmem((b ? pick(F.scene->vel[1], gu) : pick(F.scene->vel[0], gu)) + pick(S.slabs[t.slab].v_base, gu)), *v1 = gmem((b ? pick(F.scene->vel[1], gv) : pick(F.scene->vel[0], gv)) + pick(S.slabs[t.slab].v_base, gv));
        const AS_GLOBAL float *v2 = gmem((b ? S.vel[1][2] : S.vel[0][2]) + sl.v_base[2]);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int e = min(i, t.bx - 1), c = at.cell(e);
            vx[i] = v0[at.fu(e)];
            q0[i] = gmem(pick(F.scene->pd, gu) + sl.cell_base)[c];
            q1[i] = gmem(pick(F.scene->pd, gv) + sl.cell_base)[c];
            q2[i] = gmem(S.pd[2] + sl.cell_base)[c];
            yl[i] = v1[at.fv(e, 0)];
            yr[i] = v1[at.fv(e, 1)];
            zl[i] = v2[at.fw(e, 0)];
            zr[i] = v2[at.fw(e, 1)];
        }
        const float last = v0[at.fu(t.bx)];
#pragma unroll
        for (int i = 1; i <= NB; ++i)
            if (i == t.bx) vx[i] = last;
    }
    for (int s = 0; s < F.steps; ++s) {
        Column<C::cs, NB> w;
        if (F.act) {
            w.load(F.A, F.col);
            float left = w.before;
            float before = 0.f;
#pragma unroll
            for (int q = 0; q < NB / 4; ++q) {
                if (4 * q >= F.bx) continue;
                const Quad u = quad<C::cs>(F.A, F.col, F.P, q);
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * q + e;
                    const float c = w.c[i], xm = C::in_place ? left : i ? w.c[i - 1] : w.before, xp = w.c[i + 1];
                    const float4 xl = F.X[i], xr = F.X[i + 1];
                    if (i == 0) before = face_step(xl.x, xl.y, vx[0], xm, c);
                    const float after = face_step(xr.x, xr.y, vx[i + 1], c, xp);
                    q0[i] = split_step(xl.z, xl.w, q0[i], after - before);
                    vx[i] = before;
                    before = after;
                    if (e == 3) vx[i + 1] = after;
                    yl[i] = face_step(cy.l1, cy.l2, yl[i], u.yl[e], c);
                    yr[i] = face_step(cy.r1, cy.r2, yr[i], c, u.yr[e]);
                    q1[i] = split_step(cy.c3, cy.c5, q1[i], yr[i] - yl[i]);
                    zl[i] = face_step(cz.l1, cz.l2, zl[i], u.zl[e], c);
                    zr[i] = face_step(cz.r1, cz.r2, zr[i], c, u.zr[e]);
                    q2[i] = split_step(cz.c3, cz.c5, q2[i], zr[i] - zl[i]);
                    o[e] = q0[i] + q1[i] + q2[i];
                    if (C::in_place) { left = c; w.c[i] = o[e]; }
                }
                if constexpr (!C::in_place) put_quad(F.B, F.col, q, o);
            }
        }
        before_writes(F, s);
        if constexpr (C::in_place) {
            if (F.act) put_column<NB>(F.B, F.col, F.bx, w.c);
        }
        if (F.act && F.sounding() && damped != 7) {
            // (staggered scheme) on the undamped axis
            const SceneDev Z = F.scene_now();
            const ResTile u = *cmem(anew(F.tile));
            const auto w = F.across(Z, u);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                if (i >= F.bx) continue;
                const float f = F.add_sources(Z, u, w, F.step0 + s, i, 0.f);
                if (damped == 6) q0[i] += f;
                else if (damped == 5) q1[i] += f;
                else q2[i] += f;
                F.B[F.col + i] = q0[i] + q1[i] + q2[i];
            }
        }
        __syncthreads();
        F.send(s);
        F.terms(s);
        F.fetch_amp(F.step0 + s + 1);
        F.receive(s);
        F.turn();
        __syncthreads();
    }
    const SceneDev Z = F.scene_now();
    const ResTile u = *cmem(anew(F.tile));
    F.store_pressure(Z, u);
    if (!F.act) return;
    const PmlSlab zl_ = cmem(Z.slabs)[u.slab];
    const SlabAt to(zl_, u, anew(F.ly), anew(F.lz));
    const int b = (int)((F.step0 + F.steps) & 1);
    const int hu = column_axis(u), hv = across_axis(u);
    AS_GLOBAL float *v0 = gmem((b ? pick(F.scene->vel[1], hu) : pick(F.scene->vel[0], hu)) + pick(Z.slabs[u.slab].v_base, hu)), *v1 = gmem((b ? pick(F.scene->vel[1], hv) : pick(F.scene->vel[0], hv)) + pick(Z.slabs[u.slab].v_base, hv));
    AS_GLOBAL float *v2 = gmem((b ? Z.vel[1][2] : Z.vel[0][2]) + zl_.v_base[2]);
#pragma unroll
    for (int i = 0; i <= NB; ++i) {
        if (i <= u.bx) v0[to.fu(i)] = vx[i];
        if (i < NB && i < u.bx) {
            const int c = to.cell(i);
            gmem(pick(F.scene->pd, hu) + zl_.cell_base)[c] = q0[i];
            gmem(pick(F.scene->pd, hv) + zl_.cell_base)[c] = q1[i];
            gmem(Z.pd[2] + zl_.cell_base)[c] = q2[i];
            v1[to.fv(i, 0)] = yl[i];
            if (F.ly == u.by - 1) v1[to.fv(i, 1)] = yr[i];
            v2[to.fw(i, 0)] = zl[i];
            if (F.lz == u.bz - 1) v2[to.fw(i, 1)] = zr[i];
        }
    }
}

// One workgroup per tile.  No workgroup changes anything before all of its
// scene have arrived, so a scene whose workgroups cannot all be on the device
// at once (another resident launch holds it) gives the block up whole: the
// last to arrive and the first to lose patience settle it by one
// compare-and-swap on the gate.  Past the gate every neighbour is running, so
// every later wait ends.
template <int SHAPE>
__global__ __launch_bounds__(RES_THREADS, Shape<SHAPE>::waves) void resident_kernel(const ResItem *__restrict__ items, int nsteps,
                                                                                   uint32_t tag, int wait_limit, int *trouble)
{
    extern __shared__ __align__(16) float lds[];
    __shared__ int gate;
    __shared__ float4 xtab[Shape<SHAPE>::plain + 1 + Shape<SHAPE>::plain / 4];
    const ResItem it = items[blockIdx.x];
    if (!it.scene) return;
    // uniform data by way of the constant address space: scalar loads, scalar registers
    const ResScene R = *cmem(it.scene);
    const SceneDev S = *cmem(R.S);
    const ResTile t = cmem(R.tiles)[it.tile];
    u64 *clk = S.clock;
    Frame<SHAPE> F;
    F.scene = R.S;
    F.res = it.scene;
    F.tile = R.tiles + it.tile;
    F.step0 = (long long)clk[CLK_STEP];
    const long long left = (long long)clk[CLK_TARGET] - F.step0;
    if (left <= 0) return;
    F.steps = (int)min((long long)nsteps, left);
    F.tag = tag;
    F.trouble = trouble;
    F.X = xtab;
    F.A = lds;
    F.B = Shape<SHAPE>::in_place ? lds : lds + Shape<SHAPE>::lds;
    if (threadIdx.x == 0) {
        u64 expect = GATE_SHUT;
        const u64 n = __hip_atomic_fetch_add(&clk[CLK_ARRIVED], 1ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ULL;
        if (n == (u64)R.ntiles)
            __hip_atomic_compare_exchange_strong(&clk[CLK_GATE], &expect, (u64)GATE_RUN, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
    }
    F.load(S, R, t);
    if (threadIdx.x == 0) {
        u64 g;
        for (int spins = 0; (g = take_word(gmem(&clk[CLK_GATE]))) == GATE_SHUT; ++spins) {
            if (spins >= wait_limit) {
                u64 expect = GATE_SHUT;
                if (__hip_atomic_compare_exchange_strong(&clk[CLK_GATE], &expect, (u64)GATE_GIVEN_UP, __ATOMIC_RELAXED,
                                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    // with its target at its step, nothing enqueued behind this launch moves the scene
                    clk[CLK_HELD] = clk[CLK_TARGET];
                    clk[CLK_TARGET] = (u64)F.step0;
                    __hip_atomic_store(trouble, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            } else {
                __builtin_amdgcn_s_sleep(4);
            }
        }
        gate = g == GATE_RUN;
    }
    __syncthreads();
    if (!gate) return;
    // damped axes in the tile's frame
    switch (t.swap ? (t.damped & 4) | (t.damped & 1) << 1 | (t.damped >> 1 & 1) : t.damped) {
    case 0:
        if (S.inc) run_plain<SHAPE, true>(F, S, t);
        else run_plain<SHAPE, false>(F, S, t);
        break;
    case 1: run_one<SHAPE, 0>(F, S, t); break;
    case 2: run_one<SHAPE, 1>(F, S, t); break;
    case 4: run_one<SHAPE, 2>(F, S, t); break;
    default: run_more<SHAPE>(F, S, t); break;
    }
}

}  // namespace

// f(Shape<shape>, the shape's kernel)
template <class F>
static auto with_shape(int shape, F f)
{
    switch (shape) {
    case RES_FINE: return f(Shape<RES_FINE>{}, resident_kernel<RES_FINE>);
    case RES_COARSE: return f(Shape<RES_COARSE>{}, resident_kernel<RES_COARSE>);
    default: return f(Shape<RES_LARGE>{}, resident_kernel<RES_LARGE>);
    }
}

ResShape resident_shape(int shape)
{
    return with_shape(shape, [](auto c, auto) {
        using C = decltype(c);
        return ResShape{C::plain, C::one, C::more, C::cs, C::lds, C::in_place ? 1 : 2, C::words * RES_THREADS, C::recs * RES_THREADS};
    });
}

static size_t lds_bytes(int shape)
{
    const ResShape sh = resident_shape(shape);
    return sizeof(float) * (size_t)sh.buffers * (size_t)sh.lds_words;
}

int resident_capacity(int shape)
{
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    const size_t bytes = lds_bytes(shape);
    const hipError_t e = with_shape(shape, [&](auto, auto k) { return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, RES_THREADS, bytes); });
    if (e != hipSuccess) return 0;
    return per * cus;
}

hipError_t launch_resident_routes(const ResScene *scene, int ntiles, int shape, hipStream_t s)
{
    if (ntiles <= 0) return hipSuccess;
    with_shape(shape, [&](auto c, auto) {
        hipLaunchKernelGGL(route_kernel<decltype(c)::cs>, dim3(ntiles), dim3(RES_THREADS), 0, s, scene);
        return 0;
    });
    return hipGetLastError();
}

hipError_t launch_resident(int shape, const ResItem *items, int n, int nsteps, uint32_t tag, int wait_limit,
                           int *trouble, hipStream_t s, hipEvent_t done)
{
    if (n <= 0) return hipSuccess;
    const size_t bytes = lds_bytes(shape);
    with_shape(shape, [&](auto, auto k) {
        hipExtLaunchKernelGGL(k, dim3(n), dim3(RES_THREADS), bytes, s, nullptr, done, 0, items, nsteps, tag, wait_limit, trouble);
        return 0;
    });
    return hipGetLastError();
}

}  // namespace fdtd
