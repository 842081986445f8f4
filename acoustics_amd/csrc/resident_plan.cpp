// resident_plan.cpp -- which scenes run resident, how they are cut into tiles, and
// the launch lists of resident scenes.
#include "resident.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "device_scene.h"

namespace fdtd {

const char *resident_refusal(const SceneSetup &S)
{
    if (S.mac()) return "staggered scheme with face velocities";
    if (S.abc) return "Engquist boundary";
    if (S.moving) return "moving objects";
    if (S.visc) return "air viscosity";
    if (!S.cons.empty()) return "plane constraints";
    if (!S.spk.empty()) return "speaker sources";
    if (S.boundary != FDTD_BOUNDARY_RASTERIZE) return "coupled ghost cells";
    if (S.n_cpo != 1) return "acceleration noise";
    if (S.slabs.empty()) return "no PML";
    if (!S.pml_merged) return "split PML state";
    // a cell is damped along an axis exactly where that axis's segment says
    // so, and every face of a damped cell but the walls is a PML face
    for (int d = 0; d < 3; ++d) {
        for (int i = 0; i < S.n[d]; ++i)
            if ((S.cpml[d][i] != 0) == axis_plain(S, d, i) || (S.cpml[d][i] != 0) == (S.sig0[d][i] != 0))
                return "PML cells without damping";
        for (int i = 1; i < S.n[d]; ++i)
            if ((S.fpml[d][i] != 0) != (S.cpml[d][i - 1] || S.cpml[d][i])) return "PML faces off the PML cells";
        for (int i = S.inner_lo[d]; i < S.inner_hi[d]; ++i)
            if (S.f2[d][i] != S.f2[d][S.inner_lo[d]] || S.f2[d][i + 1] != S.f2[d][S.inner_lo[d]] ||
                S.f5h[d][i] != S.f5h[d][S.inner_lo[d]])
                return "uneven coefficients outside the PML";
    }
    // a record takes one object's acceleration
    for (const SpecialRec &r : S.special) {
        int obj = -1;
        for (int q = 0; q < 6; ++q) {
            if (r.gid[q] < 0) continue;
            if (obj >= 0 && S.ghosts[r.gid[q]].obj != obj) return "a cell between two objects";
            obj = S.ghosts[r.gid[q]].obj;
        }
    }
    return nullptr;
}

int ResPlan::tile_of(int i, int j, int k) const
{
    const int x[3] = {i, j, k};
    for (const ResBox &b : boxes) {
        int q[3];
        bool in = true;
        for (int d = 0; d < 3; ++d) {
            const int at = x[d] - b.lo[d];
            in = in && at >= 0 && at < b.len[d];
            q[d] = at / b.size[d];
        }
        if (in) return b.first + (q[0] * b.count[1] + q[1]) * b.count[2] + q[2];
    }
    return -1;
}

static int pieces(int len, int most) { return (len + most - 1) / most; }

// words of a tile's six faces, each face in whole lines
static int tile_words(int bx, int by, int bz)
{
    auto line = [](int n) { return (n + 15) & ~15; };
    return 2 * (line(by * bz) + line(bx * bz) + line(bx * by));
}

// LDS words from one row of columns (along z, with its two halo columns) to
// the next.  A wavefront's columns run over several rows; words after the halo
// columns make the banks go on from row to row as they do within one (16
// columns cover the 64 banks), so that its 16-byte reads do not collide.
// Tiles that fill the LDS without them do without.
static int row_pitch(const ResShape &sh, int by, int bz)
{
    const int plain = (bz + 2) * sh.column_words, even = plain + (64 - 2 * sh.column_words % 64) % 64;
    return bz % 16 && (by + 2) * even <= sh.lds_words ? even : plain;
}

// Dispatch order of a scene's tiles: eight runs, one per XCD, each an octant
// of the scene (halved along x, then y, then z, by number of tiles), so that
// most neighbours share an XCD and every XCD gets its share of the damped
// tiles; within a run the tiles with the most work first, so that the light
// ones end up beside the heavy ones on a compute unit.
static std::vector<int32_t> dispatch_order(const std::vector<ResTile> &tiles)
{
    const int n = (int)tiles.size(), per = (n + 7) / 8;
    std::vector<int32_t> o(n);
    for (int q = 0; q < n; ++q) o[q] = q;
    auto centre = [&](int q, int d) {
        const ResTile &t = tiles[q];
        if (t.swap && d < 2) d = 1 - d;
        return d == 0 ? 2 * t.i0 + t.bx : d == 1 ? 2 * t.j0 + t.by : 2 * t.k0 + t.bz;
    };
    for (int d = 0; d < 3; ++d) {
        const int runs = 8 >> d;   // runs of `per` tiles in each part to halve
        for (int part = 0; part < (1 << d); ++part) {
            const int a = std::min(n, part * runs * per), b = std::min(n, (part + 1) * runs * per);
            std::stable_sort(o.begin() + a, o.begin() + b, [&](int x, int y) { return centre(x, d) < centre(y, d); });
        }
    }
    auto weight = [&](int q) {
        const ResTile &t = tiles[q];
        const int axes = (t.damped & 1) + (t.damped >> 1 & 1) + (t.damped >> 2 & 1);
        return t.bx * (axes == 0 ? 15 : axes == 1 ? 27 : 36) + (t.re > t.rb ? 200 : 0);
    };
    for (int part = 0; part < 8; ++part)
        std::stable_sort(o.begin() + std::min(n, part * per), o.begin() + std::min(n, (part + 1) * per),
                         [&](int x, int y) { return weight(x) > weight(y); });
    return o;
}

bool resident_plan(const DeviceScene &D, int shape, ResPlan &P)
{
    const SceneSetup &S = D.S;
    const ResShape sh = resident_shape(shape);
    P = ResPlan();
    P.shape = shape;
    uint64_t words = 0;
    for (int c = 0; c < 27; ++c) {
        const int seg[3] = {c / 9, c / 3 % 3, c % 3};
        ResBox b{};
        bool some = true;
        for (int d = 0; d < 3; ++d) {
            const int cut[4] = {0, S.inner_lo[d], S.inner_hi[d], S.n[d]};
            b.lo[d] = cut[seg[d]];
            b.len[d] = cut[seg[d] + 1] - cut[seg[d]];
            if (seg[d] != 1) b.damped |= 1 << d;
            some = some && b.len[d] > 0;
        }
        if (!some) continue;
        const int axes = (b.damped & 1) + (b.damped >> 1 & 1) + (b.damped >> 2 & 1);
        const int most = axes == 0 ? sh.plain : axes == 1 ? sh.one : sh.more;
        // columns along x, or, in the shape with the longest ones, along y where a
        // sum over the axes would not come out in another order (a cell damped
        // along z only adds x, then y); edges across them: the fewest tiles, then
        // the least face per tile.  144x146x144 with an 8-cell PML takes 496 tiles
        // instead of 610, of 512; in the other shapes 2% fewer tiles gained nothing
        // (128^3 5.41 us per step against 5.29).
        int best = 1 << 30, face = 1 << 30;
        for (int swap = 0; swap < (shape == RES_LARGE && b.damped && b.damped != 4 ? 2 : 1); ++swap) {
            const int ul = b.len[swap], vl = b.len[1 - swap], u = pieces(ul, pieces(ul, most));
            for (int m = 1; m <= vl; ++m) {
                const int v = pieces(vl, m);
                int z = std::min(b.len[2], RES_COLUMNS / v);
                while (z > 1 && (tile_words(u, v, z) > sh.max_words || (v + 2) * (z + 2) * sh.column_words > sh.lds_words)) --z;
                if (z < 1 || tile_words(u, v, z) > sh.max_words) continue;
                const int mz = pieces(b.len[2], z);
                z = pieces(b.len[2], mz);
                if ((v + 2) * (z + 2) * sh.column_words > sh.lds_words) continue;
                const int n = pieces(ul, u) * pieces(vl, v) * mz;
                if (n < best || (n == best && v + z < face)) {
                    best = n;
                    face = v + z;
                    b.swap = swap;
                    b.size[swap] = u;
                    b.size[1 - swap] = v;
                    b.size[2] = z;
                }
            }
        }
        if (best == 1 << 30) return false;
        for (int d = 0; d < 3; ++d) b.count[d] = pieces(b.len[d], b.size[d]);
        b.first = (int)P.tiles.size();
        b.slab = -1;
        for (int q = 0; q < (int)S.slabs.size() && b.damped; ++q) {
            bool in = true;
            for (int d = 0; d < 3; ++d)
                in = in && b.lo[d] >= S.slabs[q].lo[d] && b.lo[d] + b.len[d] <= S.slabs[q].lo[d] + S.slabs[q].e[d];
            if (in) b.slab = q;
        }
        if (b.damped && b.slab < 0) return false;
        // one damped axis is the slab's own
        if (axes == 1 && S.slabs[b.slab].axis != (b.damped == 1 ? 0 : b.damped == 2 ? 1 : 2)) return false;
        for (int x = 0; x < b.count[0]; ++x)
            for (int y = 0; y < b.count[1]; ++y)
                for (int z = 0; z < b.count[2]; ++z) {
                    ResTile t{};
                    t.i0 = b.lo[0] + x * b.size[0];
                    t.j0 = b.lo[1] + y * b.size[1];
                    t.k0 = b.lo[2] + z * b.size[2];
                    t.bx = std::min(b.size[0], b.lo[0] + b.len[0] - t.i0);
                    t.by = std::min(b.size[1], b.lo[1] + b.len[1] - t.j0);
                    t.bz = std::min(b.size[2], b.lo[2] + b.len[2] - t.k0);
                    const int lo[3] = {t.i0, t.j0, t.k0}, hi[3] = {t.i0 + t.bx, t.j0 + t.by, t.k0 + t.bz};
                    t.swap = b.swap;
                    if (t.swap) { std::swap(t.i0, t.j0); std::swap(t.bx, t.by); }
                    t.pitch = row_pitch(sh, t.by, t.bz);
                    t.damped = b.damped;
                    t.slab = b.slab;
                    t.words = tile_words(t.bx, t.by, t.bz);
                    t.word0 = (uint32_t)words;
                    words += (uint64_t)((t.words + 16) & ~15);   // (tiles on lines of their own)
                    for (const PSrcHost &p : S.psrc) {
                        // (collocated PML cells take no source)
                        bool hit = b.damped == 0 || (S.stag_merged && axes < 3);
                        for (int d = 0; d < 3; ++d) hit = hit && lo[d] < p.hi[d] && hi[d] > p.lo[d];
                        t.src |= hit;
                    }
                    for (const SpecialBox &bx : S.boxes) {
                        bool hit = b.damped == 0;
                        for (int d = 0; d < 3; ++d) hit = hit && lo[d] < bx.hi[d] && hi[d] > bx.lo[d];
                        t.skip |= hit;
                    }
                    P.tiles.push_back(t);
                }
        P.boxes.push_back(b);
    }
    if (words > UINT32_MAX / 16) return false;   // byte offsets of both halves
    P.nwords = (uint32_t)words;
    // records and listener terms by tile
    const int sy = S.n[2], sx = S.n[1] * S.n[2];
    auto tile_of = [&](int cell) { return P.tile_of(cell / sx, cell % sx / sy, cell % sy); };
    std::vector<std::pair<int, int>> by;
    for (int r = 0; r < (int)S.special.size(); ++r) by.push_back({tile_of(S.special[r].cell), r});
    std::sort(by.begin(), by.end());
    for (const auto &e : by) {
        if (e.first < 0) return false;
        ResTile &t = P.tiles[e.first];
        if (t.damped || !t.skip) return false;
        if (t.re == t.rb) t.rb = (int)P.recs.size();
        P.recs.push_back(e.second);
        t.re = (int)P.recs.size();
        if (t.re - t.rb > sh.max_recs) return false;
    }
    by.clear();
    for (int q = 0; q < (int)S.lst_terms.size(); ++q) {
        const ListenerTerm &lt = S.lst_terms[q];
        by.push_back({tile_of(lt.kind == 0 ? lt.index : S.ghosts[lt.index].nbr), q});
    }
    std::sort(by.begin(), by.end());
    for (const auto &e : by) {
        if (e.first < 0) return false;
        ResTile &t = P.tiles[e.first];
        const ListenerTerm &lt = S.lst_terms[e.second];
        if (t.te == t.tb) t.tb = (int)P.terms.size();
        P.terms.push_back({0, e.second, lt.kind, lt.kind == 0 ? (int)D.to_dev(lt.index) : lt.index, lt.beta});
        t.te = (int)P.terms.size();
    }
    P.order = dispatch_order(P.tiles);
    return true;
}

std::string resident_check(const DeviceScene &D, int shape)
{
    const SceneSetup &S = D.S;
    if (resident_refusal(S)) return std::string();
    ResPlan P;
    if (!resident_plan(D, shape, P)) return std::string();
    const ResShape sh = resident_shape(shape);
    std::vector<uint8_t> hit((size_t)S.N, 0);
    std::vector<int> recs(S.special.size(), 0), terms(S.lst_terms.size(), 0);
    uint64_t word = 0;
    for (size_t q = 0; q < P.tiles.size(); ++q) {
        const ResTile &t = P.tiles[q];
        const int axes = (t.damped & 1) + (t.damped >> 1 & 1) + (t.damped >> 2 & 1);
        const int most = axes == 0 ? sh.plain : axes == 1 ? sh.one : sh.more;
        if (t.bx < 1 || t.by < 1 || t.bz < 1 || t.bx > most || t.by * t.bz > RES_COLUMNS) return "resident tile too large";
        if (t.pitch < (t.bz + 2) * sh.column_words || (t.by + 2) * t.pitch > sh.lds_words || t.words > sh.max_words) return "resident tile's halo too large";
        if (t.words != tile_words(t.bx, t.by, t.bz)) return "resident tile's face words";
        if (t.word0 < word || (uint64_t)t.word0 + (uint64_t)t.words > P.nwords) return "resident tiles share exchange words";
        word = (uint64_t)t.word0 + (uint64_t)t.words + 1;
        if (word > P.nwords) return "resident tile's words";
        if (t.swap && (!t.damped || t.damped == 4)) return "resident tile's columns along y";
        for (int u = t.i0; u < t.i0 + t.bx; ++u)
            for (int v = t.j0; v < t.j0 + t.by; ++v)
                for (int k = t.k0; k < t.k0 + t.bz; ++k) {
                    const int i = t.swap ? v : u, j = t.swap ? u : v;
                    if (i < 0 || j < 0 || k < 0 || i >= S.n[0] || j >= S.n[1] || k >= S.n[2]) return "resident tile outside the grid";
                    if (hit[((size_t)i * S.n[1] + j) * S.n[2] + k]++) return "a cell lies in two resident tiles";
                    const int damped = (S.cpml[0][i] ? 1 : 0) | (S.cpml[1][j] ? 2 : 0) | (S.cpml[2][k] ? 4 : 0);
                    if (damped != t.damped) return "a resident tile's class does not fit its cells";
                    if (P.tile_of(i, j, k) != (int)q) return "resident tile lookup";
                }
        for (int r = t.rb; r < t.re; ++r) ++recs[P.recs[r]];
        if (t.re - t.rb > sh.max_recs || (t.re > t.rb && (t.damped || !t.skip))) return "resident records";
        for (int r = t.tb; r < t.te; ++r) ++terms[P.terms[r].slot];
    }
    std::vector<int32_t> order(P.order);
    std::sort(order.begin(), order.end());
    for (size_t q = 0; q < order.size(); ++q)
        if (order[q] != (int32_t)q || order.size() != P.tiles.size()) return "the dispatch order does not hold every tile once";
    for (uint8_t h : hit)
        if (h != 1) return "a cell lies in no resident tile";
    for (int c : recs)
        if (c != 1) return "an object-adjacent record is not in exactly one resident tile";
    for (int c : terms)
        if (c != 1) return "a listener term is not in exactly one resident tile";
    return std::string();
}

bool ResidentScene::build(const DeviceScene &D, hipStream_t st, size_t max_bytes)
{
    release();
    if (resident_refusal(D.S)) return false;
    // (a grid that cannot fit is not cut first)
    int64_t most = 0;
    for (int shape = 0; shape < RES_SHAPES; ++shape) {
        const ResShape sh = resident_shape(shape);
        most = std::max(most, (int64_t)resident_capacity(shape) * RES_COLUMNS * std::max(sh.plain, sh.one));
    }
    if (D.S.N > most) return false;
    bool ok = false;
    for (int shape = RES_FINE; shape < RES_SHAPES && !ok; ++shape)
        ok = resident_plan(D, shape, plan) && ((int)plan.tiles.size() + 7) / 8 * 8 <= resident_capacity(shape);
    if (!ok) return false;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t b[7] = {al(sizeof(ResScene)), al(sizeof(ResTile) * plan.tiles.size()), al(sizeof(ResBox) * plan.boxes.size()),
                         al(sizeof(int32_t) * plan.recs.size()), al(sizeof(TermRef) * plan.terms.size()),
                         al(sizeof(ResRoute) * (size_t)plan.nwords), al(sizeof(unsigned long long) * 2 * (size_t)plan.nwords)};
    bytes = 0;
    for (size_t x : b) bytes += x;
    if (bytes > max_bytes) { bytes = 0; return false; }
    if (hipMalloc(&mem, bytes) != hipSuccess) {
        (void)hipGetLastError();
        mem = nullptr;
        bytes = 0;
        return false;
    }
    char *at[7];
    char *p = mem;
    for (int q = 0; q < 7; ++q) { at[q] = p; p += b[q]; }
    dev = reinterpret_cast<ResScene *>(at[0]);
    ResScene R{};
    R.S = D.self;
    R.tiles = reinterpret_cast<ResTile *>(at[1]);
    R.boxes = reinterpret_cast<ResBox *>(at[2]);
    R.recs = reinterpret_cast<int32_t *>(at[3]);
    R.terms = reinterpret_cast<TermRef *>(at[4]);
    R.route = reinterpret_cast<ResRoute *>(at[5]);
    R.words = reinterpret_cast<unsigned long long *>(at[6]);
    R.nwords = plan.nwords;
    R.ntiles = (int)plan.tiles.size();
    R.nboxes = (int)plan.boxes.size();
    // the tables in one copy
    std::vector<char> stage((size_t)(at[5] - mem), 0);
    auto put = [&](int q, const void *src, size_t n) { if (n) std::memcpy(stage.data() + (at[q] - mem), src, n); };
    put(0, &R, sizeof R);
    put(1, plan.tiles.data(), sizeof(ResTile) * plan.tiles.size());
    put(2, plan.boxes.data(), sizeof(ResBox) * plan.boxes.size());
    put(3, plan.recs.data(), sizeof(int32_t) * plan.recs.size());
    put(4, plan.terms.data(), sizeof(TermRef) * plan.terms.size());
    ok = hipMemcpyAsync(mem, stage.data(), stage.size(), hipMemcpyHostToDevice, st) == hipSuccess &&
         hipMemsetAsync(at[6], 0, b[6], st) == hipSuccess &&
         launch_resident_routes(dev, R.ntiles, plan.shape, st) == hipSuccess && hipStreamSynchronize(st) == hipSuccess;
    if (!ok) release();
    return ok;
}

void ResidentScene::release()
{
    if (mem) (void)hipFree(mem);
    mem = nullptr;
    dev = nullptr;
    bytes = 0;
}

fdtd_status ResidentProgram::upload(const std::vector<const ResidentScene *> &scenes, hipStream_t st)
{
    if (items) (void)hipFree(items);
    items = nullptr;
    n = 0;
    if (scenes.empty()) return FDTD_OK;
    std::vector<ResItem> list;
    shape = scenes[0]->plan.shape;
    // Workgroups are dispatched in list order, and a scene starts when all of
    // its own are on the device: scenes that fill the device together stand
    // next to each other (largest first, each into the first group with room).
    room = resident_capacity(shape);
    std::vector<const ResidentScene *> order(scenes);
    std::stable_sort(order.begin(), order.end(), [](const ResidentScene *a, const ResidentScene *b) {
        return a->plan.tiles.size() > b->plan.tiles.size();
    });
    std::vector<std::vector<const ResidentScene *>> groups;
    std::vector<int> used;
    for (const ResidentScene *s : order) {
        const int m = ((int)s->plan.tiles.size() + 7) / 8 * 8;
        size_t g = 0;
        while (g < groups.size() && used[g] + m > room) ++g;
        if (g == groups.size()) { groups.emplace_back(); used.push_back(0); }
        groups[g].push_back(s);
        used[g] += m;
    }
    order.clear();
    for (const auto &g : groups) order.insert(order.end(), g.begin(), g.end());
    for (const ResidentScene *s : order) {
        const int m = (int)s->plan.tiles.size(), per = (m + 7) / 8;
        // workgroup w runs on XCD w % 8 and takes the next tile of that run
        for (int w = 0; w < 8 * per; ++w) {
            const int t = (w % 8) * per + w / 8;
            list.push_back(t < m ? ResItem{s->dev, s->plan.order[t], 0} : ResItem{nullptr, 0, 0});
        }
    }
    if (!trouble) {
        FDTD_HIP_TRY(hipHostMalloc(&trouble, sizeof(int)));
        *trouble = 0;
    }
    if (!wait_limit) {
        // 7 ms, three times the longest block (256 steps of 9 us); whatever holds
        // the device for longer, another process's launch for one, sends this
        // one's scenes to the step kernels. With 230 ms, three processes that
        // solve 1000 steps at 128^3 each took 230 to 480 ms for them instead of the
        // step kernels' 16 to 44.
        const char *w = std::getenv("FDTD_RESIDENT_WAIT");
        wait_limit = w ? std::atoi(w) : 1 << 15;
    }
    FDTD_HIP_TRY(hipMalloc(&items, sizeof(ResItem) * list.size()));
    FDTD_HIP_TRY(hipMemcpyAsync(items, list.data(), sizeof(ResItem) * list.size(), hipMemcpyHostToDevice, st));
    FDTD_HIP_TRY(hipStreamSynchronize(st));
    n = (int)list.size();   // (nothing is launched before the list is there)
    return FDTD_OK;
}

// Two resident launches on different streams could each hold a part of the
// device and wait for the rest of it until both give up.  So those of one process
// that do not fit a device together follow each other there: each leaves an event,
// and a launch that does not fit beside all that other streams may still have
// running waits for them.  (Two tile shapes do not share a device by a count of
// workgroups, so they follow each other too.)  The event is the launch's own
// completion (64^3, blocks of 4 steps: 27 us a block; recorded behind it 30,
// without one 26).  A caller's stream may be under capture by then, where the
// runtime refuses to wait for its earlier events, and touching one spoils the
// capture: a stream that nobody else knows waits for a launch on such a stream at
// once, and leaves the event.
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_order;
uint64_t g_seq = 0;
// what a stream may still have running
struct Flight {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;      // of its last launch; left on `stream`, or, if that is a caller's, on the relay
    hipEvent_t handed = nullptr;    // from a caller's stream to the relay
    int n = 0, shape = -1;          // workgroups of its largest launch (0: idle); -1: of several shapes
    bool covered = false;           // another stream's launch waits for it: whoever waits for that waits for this
    uint64_t seq = 0;
};
struct Order {
    hipStream_t relay = nullptr;
    std::vector<Flight> flights;
} g_order_of[kMaxDevices];
}  // namespace

uint64_t resident_seq()
{
    std::lock_guard<std::mutex> lk(g_order);
    return g_seq;
}

void resident_idle(hipStream_t st, uint64_t seq)
{
    std::lock_guard<std::mutex> lk(g_order);
    for (Order &o : g_order_of)
        for (Flight &f : o.flights)
            if (f.stream == st && f.seq <= seq) f.n = 0;
}

void resident_forget_stream(hipStream_t st)
{
    std::lock_guard<std::mutex> lk(g_order);
    for (Order &o : g_order_of)
        for (size_t q = 0; q < o.flights.size();) {
            Flight &f = o.flights[q];
            if (f.stream != st) { ++q; continue; }
            if (f.done) (void)hipEventDestroy(f.done);
            if (f.handed) (void)hipEventDestroy(f.handed);
            o.flights.erase(o.flights.begin() + (ptrdiff_t)q);
        }
}

fdtd_status resident_reopen(const SceneDev &dev, long long *step)
{
    unsigned long long clk[CLK_WORDS];
    FDTD_HIP_TRY(hipMemcpy(clk, dev.clock, sizeof clk, hipMemcpyDeviceToHost));
    *step = (long long)clk[CLK_STEP];
    if (clk[CLK_GATE] != GATE_GIVEN_UP) return FDTD_OK;
    clk[CLK_TARGET] = clk[CLK_HELD];
    clk[CLK_ARRIVED] = 0;
    clk[CLK_GATE] = GATE_SHUT;
    FDTD_HIP_TRY(hipMemcpy(dev.clock, clk, sizeof clk, hipMemcpyHostToDevice));
    return FDTD_OK;
}

fdtd_status ResidentProgram::enqueue(hipStream_t st, int nsteps)
{
    if (n <= 0) return FDTD_OK;
    std::lock_guard<std::mutex> lk(g_order);
    int dev = 0;
    FDTD_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return FDTD_ERR_DEVICE;
    Order &order = g_order_of[dev];
    size_t own = 0;
    while (own < order.flights.size() && order.flights[own].stream != st) ++own;
    if (own == order.flights.size()) {
        Flight f;
        f.stream = st;
        FDTD_HIP_TRY(hipEventCreateWithFlags(&f.done, hipEventDisableTiming));
        FDTD_HIP_TRY(hipEventCreateWithFlags(&f.handed, hipEventDisableTiming));
        if (!order.relay) FDTD_HIP_TRY(hipStreamCreateWithFlags(&order.relay, hipStreamNonBlocking));
        order.flights.push_back(f);
    }
    int together = n;
    bool fits = true;
    for (const Flight &f : order.flights)
        if (f.stream != st && f.n) {
            together += f.n;
            fits = fits && f.shape == shape;
        }
    if (!fits || together > room)
        for (Flight &f : order.flights)
            if (f.stream != st && f.n && !f.covered) {
                FDTD_HIP_TRY(hipStreamWaitEvent(st, f.done, 0));
                f.covered = true;
            }
    Flight &f = order.flights[own];
    FDTD_HIP_TRY(launch_resident(shape, items, n, nsteps, tag, wait_limit, trouble, st, callers_stream ? f.handed : f.done));
    tag += (uint32_t)nsteps + 1;
    f.shape = f.n && f.shape != shape ? -1 : shape;
    f.n = std::max(f.n, n);
    f.covered = false;
    f.seq = ++g_seq;
    if (callers_stream) {
        FDTD_HIP_TRY(hipStreamWaitEvent(order.relay, f.handed, 0));
        FDTD_HIP_TRY(hipEventRecord(f.done, order.relay));
    }
    return FDTD_OK;
}

void ResidentProgram::release()
{
    if (items) (void)hipFree(items);
    items = nullptr;
    n = 0;
    if (trouble) (void)hipHostFree(trouble);
    trouble = nullptr;
}

}  // namespace fdtd
