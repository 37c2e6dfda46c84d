// Cell tiles: the unit of work of the kernels that evaluate faces and sum
// them into cells in one launch (host side, plain C++).
//
// A tile is a set of at most TILE_CELLS cells with every face that touches
// one of them (at most TILE_FACES: one thread each) and the cells on those
// faces' other sides, its halo (at most TILE_LOCAL cells in all).  One block
// stages the tile's cells in LDS, evaluates each face once and sums the
// results into its own cells from LDS.  A face between two tiles is evaluated
// by both, so the fewer faces a tile has per cell the better: tiles grow
// greedily, always by the cell with the most neighbours already inside, which
// gives near-cubes on hex meshes of any numbering (1.30 faces evaluated per
// face at 128^3, where perfect 4x4x4 cubes have 1.25; 1.07 on an O-grid).
//
// Only the grouping of the work depends on the tiles: a cell's sums run over
// its own six slots in order, so results do not depend on how tiles formed.
#pragma once
#include <algorithm>
#include <cstdint>
#include <exception>
#include <memory>
#include <stdexcept>
#include <thread>
#include <utility>
#include <vector>

namespace adfvm {

// 64 cells: one lane of a wave each in the cell phases.  A 4x4x4 cube has 240
// faces, so 256 threads take them in one pass at 94%.
constexpr int TILE_CELLS = 64, TILE_FACES = 256, TILE_HALO = 128, TILE_LOCAL = TILE_CELLS + TILE_HALO;

// The cells are numbered tile after tile, TILE_CELLS numbers for each tile: a
// cell's number is its position, by which the library's own arrays are laid
// out (a tile's cells are consecutive, whatever the caller's numbering; a
// tile of fewer cells leaves its last positions unused).  Every table has a
// fixed length per tile, so a block finds all of its tile's entries from its
// own index, without waiting for an offset.
//
// Local cell indices: 0 .. TILE_CELLS - 1 a tile's own cells, then its halo.
// face word: owner's local cell, neighbour's from bit 8 (0 for a ghost), kind
// byte (FACE_* and the copying-ghost bit) from bit 16, a bit for internal faces
constexpr unsigned TILE_FACE_INTERNAL = 1u << 24;
// A cell's words hold a byte per slot and two groups of six bits:
//   slots  local face; owned (bit 48); cyclic (bit 54)
//   pairs  local face paired with a cyclic slot's
//   nbr    local cell on the other side; ghost (bit 48); ghost that copies its owner (bit 54)
constexpr int TILE_BITS0 = 48, TILE_BITS1 = 54;

// The mesh as the slot tables see it ([6][nIC] arrays of the context).
struct TileMesh {
    int nIC, nIF, nF;
    const int* sFace;
    const int* sOther;             // internal cell, or -1-b for a face with a ghost
    const int* sPair;              // paired face of a cyclic slot, else -1
    const unsigned char* sFlags;   // bit 0: owned
    const unsigned char* fKind;    // [nF] kind bytes, 0 for internal faces
    unsigned copyBit;              // the kind byte's copying-ghost bit
};

// Vectors whose new entries are not set to zero: their memory is first touched
// by the threads that fill it.
template <typename T> struct Unset : std::allocator<T> {
    template <typename U> struct rebind { typedef Unset<U> other; };
    template <typename U> void construct(U* p) noexcept { ::new ((void*)p) U; }
    template <typename U, typename... A> void construct(U* p, A&&... a) { ::new ((void*)p) U(std::forward<A>(a)...); }
};
template <typename T> using Buffer = std::vector<T, Unset<T>>;

struct Tiles {
    int n = 0;                         // tiles
    Buffer<int> toUser;                // [n][TILE_CELLS] position -> caller's cell, ~(a cell of the tile) if unused
    Buffer<int> toTile;                // caller's cell -> position
    Buffer<int> halo;                  // [n][TILE_HALO] positions; unused entries repeat the tile's first cell
    Buffer<int> faceId;                // [n][TILE_FACES] global face; unused entries repeat the first
    Buffer<unsigned> face;             // [n][TILE_FACES] face words; unused entries are an internal face of cell 0
    Buffer<uint64_t> slots, pairs, nbr;   // [n][TILE_CELLS] cell words
};

// The parts over_threads splits [0, n) into: at most 8, each of `grain` entries
// or more.
inline int thread_parts(int n, int grain) {
    return std::max(1, std::min({8, (int)std::thread::hardware_concurrency(), n / grain}));
}

// f(a, b, k) over the parts k of [0, n), a host thread each; a part whose
// thread cannot be started runs on this one, and the first exception of any
// part is rethrown here when all have ended.  A thread takes about 30 us to
// start, and now and then 3 ms where the host's cores are taken (seen with 70 tiles in
// four threads), so `grain` entries should take several 100 us.
template <typename F> void over_threads(int n, int grain, F&& f) {
    const int nt = thread_parts(n, grain);
    if (nt == 1) {
        f(0, n, 0);
        return;
    }
    std::vector<std::exception_ptr> err(nt);
    auto part = [&](int k) {
        try {
            f((int)((long)n * k / nt), (int)((long)n * (k + 1) / nt), k);
        } catch (...) {
            err[k] = std::current_exception();
        }
    };
    std::vector<std::thread> th;
    th.reserve(nt);
    for (int k = 1; k < nt; k++) {
        try {
            th.emplace_back(part, k);
        } catch (...) {
            part(k);
        }
    }
    part(0);
    for (auto& x : th) x.join();
    for (auto& e : err)
        if (e) std::rethrow_exception(e);
}
constexpr int CELL_GRAIN = 8192, TILE_GRAIN = 96;

// The cells' slots, six entries a cell: the other cell, or -2 - cell across a
// cyclic face, or -1 (a ghost); the face, or ~face where the cell is not its
// owner.  The slot tables are rows of all cells, six cache lines for a cell.
struct CellSlots {
    Buffer<int> near, face;
};
inline CellSlots cell_slots(const TileMesh& m) {
    const long n = m.nIC;
    CellSlots cell;
    cell.near.resize(6 * n);
    cell.face.resize(6 * n);
    over_threads(m.nIC, CELL_GRAIN, [&](int a, int b, int) {
        for (long c = a; c < b; c++)
            for (int j = 0; j < 6; j++) {
                const long s = j * n + c;
                const int o = m.sOther[s], f = m.sFace[s];
                cell.near[6 * c + j] = o < 0 ? -1 : f >= m.nIF && m.sPair[s] >= 0 ? -2 - o : o;
                cell.face[6 * c + j] = m.sFlags[s] & 1 ? f : ~f;
            }
    });
    return cell;
}

// Grows the tiles: tileOf order as lists of own cells, ascending in each.
// Candidates wait in one queue per number of neighbours inside (oldest
// first); stale entries are skipped when they come up.
// A cell waits for its neighbours' cache lines, so its state is 8 bytes.
inline void grow_tiles(const TileMesh& m, const CellSlots& cell, std::vector<int>& cells, std::vector<int>& start) {
    const long n = m.nIC;
    struct State {
        int gain = 0;                  // 8 tile + the neighbours inside the last tile it was a candidate of; -1: in a tile
        int at = -1;                   // 2 tile of the last tile it was beside, or that + 1: inside it
    };
    std::vector<State> state(n);
    int queue[7][6 * TILE_CELLS], head[7], tail[7];      // a cell of the tile adds at most six entries
    cells.clear();
    cells.reserve(n);
    start.assign(1, 0);
    long seed = 0;
    while ((long)cells.size() < n) {
        const int tile = (int)start.size() - 1;
        const size_t first = cells.size();
        int faces = 0, halo = 0;
        for (int g = 1; g <= 6; g++) head[g] = tail[g] = 0;
        for (;;) {
            int c = -1;
            for (int g = 6; g >= 1 && c < 0; g--)
                while (head[g] < tail[g]) {
                    const int k = queue[g][head[g]];
                    if (state[k].gain != 8 * tile + g) { head[g]++; continue; }
                    c = k;
                    break;
                }
            if (c < 0) {               // a new tile, or a region the tile has used up: the first cell left
                while (seed < n && state[seed].gain < 0) seed++;
                if (seed == n) break;
                c = (int)seed;
            }
            // faces and halo cells the tile would have with c
            const int* near = &cell.near[6L * c];
            int df = 0, dh = state[c].at == 2 * tile ? -1 : 0;
            int fresh[6], nFresh = 0;
            for (int j = 0; j < 6; j++) {
                const int e = near[j], o = e < -1 ? -2 - e : e;
                const int at = o < 0 ? 2 * tile : state[o].at;
                if (e < -1) df += 2;
                else if (at != 2 * tile + 1) df += 1;
                if (at < 2 * tile && o != c) {
                    bool seen = false;
                    for (int k = 0; k < nFresh; k++) seen = seen || fresh[k] == o;
                    if (!seen) { fresh[nFresh++] = o; dh++; }
                }
            }
            const int own = (int)(cells.size() - first) + 1;
            if (own > 1 && (own > TILE_CELLS || faces + df > TILE_FACES || halo + dh > TILE_HALO)) break;
            faces += df;
            halo += dh;
            state[c].gain = -1;
            state[c].at = 2 * tile + 1;
            cells.push_back(c);
            for (int k = 0; k < nFresh; k++) state[fresh[k]].at = 2 * tile;
            for (int j = 0; j < 6; j++) {
                const int o = near[j];
                if (o < 0 || state[o].gain < 0) continue;
                const int g = std::max(state[o].gain, 8 * tile) + 1;
                state[o].gain = g;
                queue[g & 7][tail[g & 7]++] = o;
            }
        }
        std::sort(cells.begin() + first, cells.end());
        start.push_back((int)cells.size());
    }
}

// Reorders the tiles (cells, start as grow_tiles leaves them) so that tiles
// near one another in the mesh are near in the order at every scale: tiles
// are joined into groups of up to 8, always by the tile with the most shared
// faces, the groups into groups of groups, and so on, and read off group by
// group.  The tiles a chip die works on at one time then share their halos
// through its cache.  In growth order a layer of tiles spans the whole mesh
// before the next begins, and every halo came from memory: at 128^3 FP32 the
// four kernels of a stage and its reverse read 3.92 GB, in this order 3.01 GB.
inline void order_tiles(const TileMesh& m, const CellSlots& cell, std::vector<int>& cells,
                        std::vector<int>& start) {
    const long n = m.nIC;
    const int nt = (int)start.size() - 1;
    Buffer<int> node(n);                             // cell -> tile
    over_threads(nt, 8 * TILE_GRAIN, [&](int a, int b, int) {
        for (int t = a; t < b; t++)
            for (int i = start[t]; i < start[t + 1]; i++) node[cells[i]] = t;
    });
    // edges between the nodes of a level, by their first node, then by the other
    struct Edge { int b, w; };
    std::vector<Edge> edges;
    std::vector<int> first(nt + 1, 0);               // a node's edges
    auto by_node = [](const Edge& x, const Edge& y) { return x.b < y.b; };
    {
        const int np = thread_parts(nt, 4 * TILE_GRAIN);
        std::vector<std::vector<Edge>> part(np);
        over_threads(nt, 4 * TILE_GRAIN, [&](int a, int b, int p) {
            std::vector<Edge>& e = part[p];
            std::vector<int> at(nt, -1);             // a tile's edge
            e.reserve(16 * (size_t)(b - a));
            for (int t = a; t < b; t++) {
                const int e0 = (int)e.size();
                for (int i = start[t]; i < start[t + 1]; i++)
                    for (int j = 0; j < 6; j++) {
                        const int x = cell.near[6L * cells[i] + j];
                        const int o = x < -1 ? -2 - x : x, k = o < 0 ? t : node[o];
                        if (k == t) continue;
                        if (at[k] < e0) { at[k] = (int)e.size(); e.push_back({k, 0}); }
                        e[at[k]].w++;
                    }
                std::sort(e.begin() + e0, e.end(), by_node);
                first[t + 1] = (int)e.size() - e0;
            }
        });
        for (const auto& e : part) edges.insert(edges.end(), e.begin(), e.end());
        for (int t = 0; t < nt; t++) first[t + 1] += first[t];
    }
    // the tiles in order, node by node: node k's begin at leaf[k]
    std::vector<int> order(nt), leaf(nt + 1);
    for (int t = 0; t < nt; t++) order[t] = leaf[t] = t;
    leaf[nt] = nt;
    for (int nodes = nt; nodes > 1;) {
        std::vector<int> group(nodes, -1), weight(nodes, 0), mark(nodes, -1), beside, order2, leaf2(1, 0);
        std::vector<int> member, from(1, 0);         // the groups' nodes
        order2.reserve(nt);
        for (int seed = 0; seed < nodes; seed++) {
            if (group[seed] >= 0) continue;
            const int g = (int)leaf2.size() - 1;
            beside.clear();
            for (int c = seed, size = 0; c >= 0 && size < 8; size++) {
                group[c] = g;
                member.push_back(c);
                order2.insert(order2.end(), order.begin() + leaf[c], order.begin() + leaf[c + 1]);
                for (int e = first[c]; e < first[c + 1]; e++) {
                    const int o = edges[e].b;
                    if (group[o] >= 0) continue;
                    if (mark[o] != g) { mark[o] = g; weight[o] = 0; beside.push_back(o); }
                    weight[o] += edges[e].w;
                }
                c = -1;
                for (int o : beside)
                    if (group[o] < 0 && (c < 0 || weight[o] > weight[c])) c = o;
            }
            leaf2.push_back((int)order2.size());
            from.push_back((int)member.size());
        }
        const int up = (int)leaf2.size() - 1;
        const bool joined = up < nodes;
        order.swap(order2);
        leaf.swap(leaf2);
        if (!joined) break;                          // separate regions only
        // the groups' edges: their nodes', one per pair, weights added
        std::vector<Edge> edges2;
        std::vector<int> first2(1, 0), at(up, -1);
        for (int g = 0; g < up; g++) {
            const int e0 = (int)edges2.size();
            for (int k = from[g]; k < from[g + 1]; k++)
                for (int e = first[member[k]]; e < first[member[k] + 1]; e++) {
                    const int o = group[edges[e].b];
                    if (o == g) continue;
                    if (at[o] < e0) { at[o] = (int)edges2.size(); edges2.push_back({o, 0}); }
                    edges2[at[o]].w += edges[e].w;
                }
            std::sort(edges2.begin() + e0, edges2.end(), by_node);
            first2.push_back((int)edges2.size());
        }
        edges.swap(edges2);
        first.swap(first2);
        nodes = up;
    }
    std::vector<int> cells2, start2(1, 0);
    cells2.reserve(n);
    for (int t : order) {
        cells2.insert(cells2.end(), cells.begin() + start[t], cells.begin() + start[t + 1]);
        start2.push_back((int)cells2.size());
    }
    cells.swap(cells2);
    start.swap(start2);
}

// A set of positions by open addressing, at most half full.
struct PositionSet {
    static constexpr int SIZE = 256;
    static_assert(2 * TILE_HALO <= SIZE && SIZE == 1 << (32 - 24), "half full; the hash's range");
    int key[SIZE];
    void clear() { std::fill(key, key + SIZE, -1); }
    int find(int p) const {            // p's entry, or the free one where it goes
        unsigned h = (unsigned)p * 2654435761u >> 24;
        while (key[h] != -1 && key[h] != p) h = (h + 1) & (SIZE - 1);
        return (int)h;
    }
};

// Lists a tile and writes its words.  Faces in order: the cells' internal and
// cyclic faces as their slots come, the paired faces of cyclic slots (whose
// neighbour side the cell takes), the faces with a ghost by kind.  A tile has at
// most TILE_FACES faces and TILE_HALO halo cells.
// An internal face's second slot, and a paired face that an own cell owns, are
// found among the six faces of the cell across; every other face is a new one.
inline void fill_tile(const TileMesh& m, const CellSlots& cell, int tile, int nOwn, Tiles& out) {
    const long n = m.nIC;
    const size_t c0 = (size_t)tile * TILE_CELLS, f0 = (size_t)tile * TILE_FACES;
    int* halo = out.halo.data() + (size_t)tile * TILE_HALO;
    int* id = out.faceId.data() + f0;
    unsigned* word = out.face.data() + f0;
    const int* own = out.toUser.data() + c0;
    struct { int near[6], face[6]; } cs[TILE_CELLS];
    int at[TILE_CELLS][6];             // the position across (-1: a ghost)
    unsigned char local[TILE_CELLS][6], number[TILE_CELLS][6], pair[TILE_CELLS][6];     // local cell, face, paired face
    struct Ghost { int f, i, j; unsigned char kind; } ghost[TILE_FACES];
    PositionSet halos;
    uint64_t found[TILE_HALO];         // halo cells: position, entry of the set (8 bits)
    unsigned char byEntry[PositionSet::SIZE];
    int nFace = 0, nHalo = 0, nGhost = 0;
    bool pairs = false;
    halos.clear();
    for (int i = 0; i < nOwn; i++) {
        std::copy_n(&cell.near[6L * own[i]], 6, cs[i].near);
        std::copy_n(&cell.face[6L * own[i]], 6, cs[i].face);
        for (int j = 0; j < 6; j++) {
            const int e = cs[i].near[j];
            local[i][j] = pair[i][j] = 0;
            if (e == -1) {
                const int f = cs[i].face[j] < 0 ? ~cs[i].face[j] : cs[i].face[j];
                at[i][j] = -1;
                ghost[nGhost++] = {f, i, j, m.fKind[f]};
                continue;
            }
            pairs = pairs || e < -1;
            const int p = at[i][j] = out.toTile[e < -1 ? -2 - e : e];
            if (p / TILE_CELLS == tile) {
                local[i][j] = (unsigned char)(p % TILE_CELLS);
                continue;
            }
            const int h = halos.find(p);
            local[i][j] = (unsigned char)h;          // a local cell below
            if (halos.key[h] == -1) {
                halos.key[h] = p;
                found[nHalo++] = (uint64_t)p << 8 | (unsigned)h;
            }
        }
    }
    std::sort(found, found + nHalo);
    for (int k = 0; k < nHalo; k++) {
        halo[k] = (int)(found[k] >> 8);
        byEntry[found[k] & 255] = (unsigned char)(TILE_CELLS + k);
    }
    // the face of own cell o (whose faces up to there are numbered) that is f, or -1
    auto numbered = [&](int o, int last, int f) {
        for (int q = 0; q < last; q++)
            if (at[o][q] >= 0 && (cs[o].face[q] == f || cs[o].face[q] == ~f)) return (int)number[o][q];
        return -1;
    };
    for (int i = 0; i < nOwn; i++)
        for (int j = 0; j < 6; j++) {
            const int p = at[i][j];
            if (p < 0) continue;
            const int f = cs[i].face[j] < 0 ? ~cs[i].face[j] : cs[i].face[j];
            int k = -1;
            if (p / TILE_CELLS != tile) local[i][j] = byEntry[local[i][j]];
            else if (f < m.nIF && local[i][j] <= i) k = numbered(local[i][j], local[i][j] < i ? 6 : j, f);
            if (k < 0) { k = nFace; id[nFace++] = f; }
            number[i][j] = (unsigned char)k;
        }
    if (pairs)
        for (int i = 0; i < nOwn; i++)
            for (int j = 0; j < 6; j++) {
                if (cs[i].near[j] >= -1) continue;
                const int g = m.sPair[j * n + own[i]];
                int k = at[i][j] / TILE_CELLS == tile ? numbered(local[i][j], 6, g) : -1;
                if (k < 0) { k = nFace; id[nFace++] = g; }
                pair[i][j] = (unsigned char)k;
            }
    std::sort(ghost, ghost + nGhost, [](const Ghost& a, const Ghost& b) {
        return a.kind != b.kind ? a.kind < b.kind : a.f < b.f;
    });
    for (int k = 0; k < nGhost; k++) {
        number[ghost[k].i][ghost[k].j] = (unsigned char)nFace;
        id[nFace++] = ghost[k].f;
    }
    std::fill(id + nFace, id + TILE_FACES, id[0]);
    std::fill(word + nFace, word + TILE_FACES, 0u);
    std::fill(halo + nHalo, halo + TILE_HALO, (int)c0);
    for (int i = 0; i < nOwn; i++) {
        uint64_t sl = 0, pr = 0, nb = 0;
        for (int j = 0; j < 6; j++) {
            const bool isOwn = cs[i].face[j] >= 0;
            const int f = isOwn ? cs[i].face[j] : ~cs[i].face[j], lf = number[i][j];
            const unsigned lo = local[i][j], kind = f < m.nIF ? 0u : m.fKind[f];
            if (at[i][j] < 0) {
                nb |= 1ull << (TILE_BITS0 + j);
                if (kind & m.copyBit) nb |= 1ull << (TILE_BITS1 + j);
            }
            sl |= (uint64_t)lf << (8 * j);
            nb |= (uint64_t)lo << (8 * j);
            if (isOwn) sl |= 1ull << (TILE_BITS0 + j);
            word[lf] = (isOwn ? (unsigned)i | lo << 8 : lo | (unsigned)i << 8) | kind << 16 |
                       (f < m.nIF ? TILE_FACE_INTERNAL : 0u);
            if (cs[i].near[j] < -1) {
                const int lg = pair[i][j];
                sl |= 1ull << (TILE_BITS1 + j);
                pr |= (uint64_t)lg << (8 * j);
                word[lg] = lo | (unsigned)i << 8 | (unsigned)m.fKind[id[lg]] << 16;
            }
        }
        out.slots[c0 + i] = sl;
        out.pairs[c0 + i] = pr;
        out.nbr[c0 + i] = nb;
    }
    for (int i = nOwn; i < TILE_CELLS; i++) out.slots[c0 + i] = out.pairs[c0 + i] = out.nbr[c0 + i] = 0;
}

inline void build_tiles(const TileMesh& m, Tiles& t) {
    const CellSlots cell = cell_slots(m);
    std::vector<int> cells, start;
    grow_tiles(m, cell, cells, start);
    order_tiles(m, cell, cells, start);
    t.n = (int)start.size() - 1;
    const size_t nPos = (size_t)t.n * TILE_CELLS, nFaces = (size_t)t.n * TILE_FACES;
    if (nFaces > 0x7fffffffu) throw std::length_error("mesh too large for 32-bit tile lists");
    t.toUser.resize(nPos);
    t.toTile.resize(m.nIC);
    t.halo.resize((size_t)t.n * TILE_HALO);
    t.faceId.resize(nFaces);
    t.face.resize(nFaces);
    t.slots.resize(nPos);
    t.pairs.resize(nPos);
    t.nbr.resize(nPos);
    over_threads(t.n, 8 * TILE_GRAIN, [&](int a, int b, int) {
        for (int k = a; k < b; k++)
            for (int i = 0; i < TILE_CELLS; i++) {
                const bool used = start[k] + i < start[k + 1];
                const int c = cells[start[k] + (used ? i : 0)];
                t.toUser[(size_t)k * TILE_CELLS + i] = used ? c : ~c;
                if (used) t.toTile[c] = k * TILE_CELLS + i;
            }
    });
    over_threads(t.n, TILE_GRAIN, [&](int a, int b, int) {
        for (int k = a; k < b; k++) fill_tile(m, cell, k, start[k + 1] - start[k], t);
    });
}

}  // namespace adfvm
