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
#include <stdexcept>
#include <system_error>
#include <thread>
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
    const unsigned char* fKind;    // [nF] kind bytes
    unsigned copyBit;              // the kind byte's copying-ghost bit
};

struct Tiles {
    int n = 0;                         // tiles
    std::vector<int> toUser;           // [n][TILE_CELLS] position -> caller's cell, ~(a cell of the tile) if unused
    std::vector<int> toTile;           // caller's cell -> position
    std::vector<int> halo;             // [n][TILE_HALO] positions; unused entries repeat the tile's first cell
    std::vector<int> faceId;           // [n][TILE_FACES] global face; unused entries repeat the first
    std::vector<unsigned> face;        // [n][TILE_FACES] face words; unused entries are an internal face of cell 0
    std::vector<uint64_t> slots, pairs, nbr;   // [n][TILE_CELLS] cell words
};

// The parts over_threads splits [0, n) into.
inline int thread_parts(int n) { return std::max(1, std::min({8, (int)std::thread::hardware_concurrency(), n / 64})); }

// f(a, b, k) over the parts k of [0, n), a host thread each; a part whose
// thread cannot be started runs on this one, and the first exception of any
// part is rethrown here when all have ended.
template <typename F> void over_threads(int n, F&& f) {
    const int nt = thread_parts(n);
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
        } catch (const std::system_error&) {
            part(k);
        }
    }
    part(0);
    for (auto& x : th) x.join();
    for (auto& e : err)
        if (e) std::rethrow_exception(e);
}

// A cell's six neighbours in one place, n cells: the other cell, or -2 - cell
// across a cyclic face, or -1 (a ghost).  The slot tables are rows of all
// cells, six cache lines for a cell.
inline std::vector<int> neighbour_list(const TileMesh& m) {
    const long n = m.nIC;
    std::vector<int> near(6 * n);
    over_threads(m.nIC, [&](int a, int b, int) {
        for (long c = a; c < b; c++)
            for (int j = 0; j < 6; j++) {
                const int o = m.sOther[j * n + c];
                near[6 * c + j] = o < 0 ? -1 : m.sPair[j * n + c] >= 0 ? -2 - o : o;
            }
    });
    return near;
}

// Grows the tiles: tileOf order as lists of own cells, ascending in each.
// Candidates wait in one queue per number of neighbours inside (oldest
// first); stale entries are skipped when they come up.
inline void grow_tiles(const TileMesh& m, const std::vector<int>& near, std::vector<int>& cells,
                       std::vector<int>& start) {
    const long n = m.nIC;
    std::vector<char> taken(n, 0);
    std::vector<int> gain(n, 0), gainTile(n, -1), nearTile(n, -1);
    std::vector<int> queue[7];
    size_t head[7];
    cells.clear();
    cells.reserve(n);
    start.assign(1, 0);
    long seed = 0;
    while ((long)cells.size() < n) {
        const int tile = (int)start.size() - 1;
        const size_t first = cells.size();
        int faces = 0, halo = 0;
        for (int g = 1; g <= 6; g++) { queue[g].clear(); head[g] = 0; }
        for (;;) {
            int c = -1;
            for (int g = 6; g >= 1 && c < 0; g--)
                while (head[g] < queue[g].size()) {
                    const int k = queue[g][head[g]];
                    if (taken[k] || gain[k] != g) { head[g]++; continue; }
                    c = k;
                    break;
                }
            if (c < 0) {               // a new tile, or a region the tile has used up: the first cell left
                while (seed < n && taken[seed]) seed++;
                if (seed == n) break;
                c = (int)seed;
            }
            // faces and halo cells the tile would have with c
            int df = 0, dh = nearTile[c] == tile ? -1 : 0;
            int fresh[6], nFresh = 0;
            for (int j = 0; j < 6; j++) {
                const int e = near[6L * c + j], o = e < -1 ? -2 - e : e;
                if (e < -1) df += 2;
                else if (o < 0) df += 1;
                else if (nearTile[o] != -2 - tile) df += 1;
                if (o >= 0 && o != c && nearTile[o] != tile && nearTile[o] != -2 - tile) {
                    bool seen = false;
                    for (int k = 0; k < nFresh; k++) seen = seen || fresh[k] == o;
                    if (!seen) { fresh[nFresh++] = o; dh++; }
                }
            }
            const int own = (int)(cells.size() - first) + 1;
            if (own > 1 && (own > TILE_CELLS || faces + df > TILE_FACES || halo + dh > TILE_HALO)) break;
            faces += df;
            halo += dh;
            taken[c] = 1;
            gainTile[c] = tile;
            nearTile[c] = -2 - tile;               // inside
            cells.push_back(c);
            for (int k = 0; k < nFresh; k++) nearTile[fresh[k]] = tile;
            for (int j = 0; j < 6; j++) {
                const int o = near[6L * c + j];
                if (o < 0 || taken[o]) continue;
                if (gainTile[o] != tile) { gainTile[o] = tile; gain[o] = 0; }
                queue[++gain[o]].push_back(o);
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
inline void order_tiles(const TileMesh& m, const std::vector<int>& near, std::vector<int>& cells,
                        std::vector<int>& start) {
    const long n = m.nIC;
    int nodes = (int)start.size() - 1;
    const int nt = nodes;
    std::vector<int> node(n);                        // cell -> tile
    for (int t = 0; t < nt; t++)
        for (int i = start[t]; i < start[t + 1]; i++) node[cells[i]] = t;
    struct Edge { int a, b, w; };
    auto merge = [](std::vector<Edge>& e) {          // one edge per pair, weights added
        std::sort(e.begin(), e.end(), [](const Edge& x, const Edge& y) { return x.a != y.a ? x.a < y.a : x.b < y.b; });
        size_t k = 0;
        for (size_t i = 0; i < e.size(); i++) {
            if (k && e[k - 1].a == e[i].a && e[k - 1].b == e[i].b) e[k - 1].w += e[i].w;
            else e[k++] = e[i];
        }
        e.resize(k);
    };
    std::vector<Edge> edges;
    std::vector<std::vector<Edge>> part(thread_parts(nt));
    over_threads(nt, [&](int a, int b, int p) {
        std::vector<Edge>& e = part[p];
        for (int t = a; t < b; t++) {
            const size_t first = e.size();
            for (int i = start[t]; i < start[t + 1]; i++)
                for (int j = 0; j < 6; j++) {
                    const int x = near[6L * cells[i] + j], o = x < -1 ? -2 - x : x;
                    if (o < 0 || node[o] == t) continue;
                    bool seen = false;
                    for (size_t k = first; k < e.size() && !seen; k++)
                        if (e[k].b == node[o]) { e[k].w++; seen = true; }
                    if (!seen) e.push_back({t, node[o], 1});
                }
        }
    });
    for (const auto& e : part) edges.insert(edges.end(), e.begin(), e.end());
    std::vector<std::vector<int>> leaves(nt);        // a node's tiles in order
    for (int t = 0; t < nt; t++) leaves[t] = {t};
    while (nodes > 1) {
        merge(edges);
        std::vector<int> first(nodes + 1, 0), group(nodes, -1), weight(nodes, 0), mark(nodes, -1), beside;
        for (const Edge& e : edges) first[e.a + 1]++;
        for (int k = 0; k < nodes; k++) first[k + 1] += first[k];
        std::vector<std::vector<int>> up;
        for (int seed = 0; seed < nodes; seed++) {
            if (group[seed] >= 0) continue;
            const int g = (int)up.size();
            up.emplace_back();
            beside.clear();
            for (int c = seed, size = 0; c >= 0 && size < 8; size++) {
                group[c] = g;
                up[g].insert(up[g].end(), leaves[c].begin(), leaves[c].end());
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
        }
        const bool joined = (int)up.size() < nodes;
        nodes = (int)up.size();
        leaves.swap(up);
        if (!joined) break;                          // separate regions only
        size_t k = 0;
        for (const Edge& e : edges)
            if (group[e.a] != group[e.b]) edges[k++] = {group[e.a], group[e.b], e.w};
        edges.resize(k);
    }
    std::vector<int> cells2, start2(1, 0);
    cells2.reserve(n);
    for (const auto& l : leaves)
        for (int t : l) {
            cells2.insert(cells2.end(), cells.begin() + start[t], cells.begin() + start[t + 1]);
            start2.push_back((int)cells2.size());
        }
    cells.swap(cells2);
    start.swap(start2);
}

// Numbers small integers in the order they are first given (open addressing;
// at most half full).
struct Numbering {
    static constexpr int SIZE = 1024;
    int key[SIZE], value[SIZE];
    void clear() { std::fill(key, key + SIZE, -1); }
    int* find(int k) {                 // k's entry, or the free one where it goes
        unsigned h = (unsigned)k * 2654435761u >> 22;
        while (key[h] != -1 && key[h] != k) h = (h + 1) & (SIZE - 1);
        return &key[h];
    }
    int at(int k) { return value[find(k) - key]; }
    bool add(int k, int v) {           // false: k is there already
        int* p = find(k);
        if (*p == k) return false;
        *p = k;
        value[p - key] = v;
        return true;
    }
};

// Lists a tile and writes its words.  Faces in order: the cells' internal and
// cyclic faces as their slots come, the paired faces of cyclic slots (whose
// neighbour side the cell takes), the faces with a ghost by kind.  A tile has at
// most TILE_FACES faces and TILE_HALO halo cells.
inline void fill_tile(const TileMesh& m, int tile, int nOwn, Numbering& faces, Numbering& cells, Tiles& out) {
    const long n = m.nIC;
    const size_t c0 = (size_t)tile * TILE_CELLS, f0 = (size_t)tile * TILE_FACES;
    int* halo = out.halo.data() + (size_t)tile * TILE_HALO;
    int* id = out.faceId.data() + f0;
    unsigned* word = out.face.data() + f0;
    const int* own = out.toUser.data() + c0;
    int face[TILE_CELLS][6], other[TILE_CELLS][6], ghost[TILE_FACES];
    int nFace = 0, nHalo = 0, nGhost = 0;
    bool pairs = false;
    faces.clear();
    cells.clear();
    for (int j = 0; j < 6; j++)
        for (int i = 0; i < nOwn; i++) {
            face[i][j] = m.sFace[j * n + own[i]];
            other[i][j] = m.sOther[j * n + own[i]];
        }
    for (int i = 0; i < nOwn; i++)
        for (int j = 0; j < 6; j++) {
            const int f = face[i][j], o = other[i][j];
            if (o < 0) {
                ghost[nGhost++] = f;
                continue;
            }
            if (faces.add(f, nFace)) id[nFace++] = f;
            pairs = pairs || f >= m.nIF;
            const int p = out.toTile[o];
            if (p / TILE_CELLS != tile && cells.add(p, 0)) halo[nHalo++] = p;
        }
    std::sort(halo, halo + nHalo);
    for (int k = 0; k < nHalo; k++) cells.value[cells.find(halo[k]) - cells.key] = TILE_CELLS + k;
    if (pairs)
        for (int i = 0; i < nOwn; i++)
            for (int j = 0; j < 6; j++) {
                const int g = m.sPair[j * n + own[i]];
                if (g >= 0 && faces.add(g, nFace)) id[nFace++] = g;
            }
    std::sort(ghost, ghost + nGhost, [&](int a, int b) {
        return m.fKind[a] != m.fKind[b] ? m.fKind[a] < m.fKind[b] : a < b;
    });
    for (int k = 0; k < nGhost; k++)
        if (faces.add(ghost[k], nFace)) id[nFace++] = ghost[k];
    std::fill(id + nFace, id + TILE_FACES, id[0]);
    std::fill(halo + nHalo, halo + TILE_HALO, (int)c0);
    for (int i = 0; i < nOwn; i++) {
        uint64_t sl = 0, pr = 0, nb = 0;
        for (int j = 0; j < 6; j++) {
            const long s = j * n + own[i];
            const int f = face[i][j], o = other[i][j];
            const bool isOwn = m.sFlags[s] & 1;
            const int lf = faces.at(f);
            unsigned lo = 0;
            if (o >= 0) {
                const int p = out.toTile[o];
                lo = p / TILE_CELLS == tile ? p % TILE_CELLS : cells.at(p);
            } else {
                nb |= 1ull << (TILE_BITS0 + j);
                if (m.fKind[f] & m.copyBit) nb |= 1ull << (TILE_BITS1 + j);
            }
            sl |= (uint64_t)lf << (8 * j);
            nb |= (uint64_t)lo << (8 * j);
            if (isOwn) sl |= 1ull << (TILE_BITS0 + j);
            word[lf] = (isOwn ? (unsigned)i | lo << 8 : lo | (unsigned)i << 8) | (unsigned)m.fKind[f] << 16 |
                       (f < m.nIF ? TILE_FACE_INTERNAL : 0u);
            const int g = f >= m.nIF ? m.sPair[s] : -1;
            if (g >= 0) {
                const int lg = faces.at(g);
                sl |= 1ull << (TILE_BITS1 + j);
                pr |= (uint64_t)lg << (8 * j);
                word[lg] = lo | (unsigned)i << 8 | (unsigned)m.fKind[g] << 16;
            }
        }
        out.slots[c0 + i] = sl;
        out.pairs[c0 + i] = pr;
        out.nbr[c0 + i] = nb;
    }
}

inline void build_tiles(const TileMesh& m, Tiles& t) {
    std::vector<int> cells, start;
    {
        const std::vector<int> near = neighbour_list(m);
        grow_tiles(m, near, cells, start);
        order_tiles(m, near, cells, start);
    }
    t.n = (int)start.size() - 1;
    const size_t nPos = (size_t)t.n * TILE_CELLS, nFaces = (size_t)t.n * TILE_FACES;
    if (nFaces > 0x7fffffffu) throw std::length_error("mesh too large for 32-bit tile lists");
    t.toUser.resize(nPos);
    t.toTile.resize(m.nIC);
    for (int k = 0; k < t.n; k++)
        for (int i = 0; i < TILE_CELLS; i++) {
            const bool used = start[k] + i < start[k + 1];
            const int c = cells[start[k] + (used ? i : 0)];
            t.toUser[(size_t)k * TILE_CELLS + i] = used ? c : ~c;
            if (used) t.toTile[c] = k * TILE_CELLS + i;
        }
    t.halo.resize((size_t)t.n * TILE_HALO);
    t.faceId.resize(nFaces);
    t.face.assign(nFaces, 0);
    t.slots.assign(nPos, 0);
    t.pairs.assign(nPos, 0);
    t.nbr.assign(nPos, 0);
    over_threads(t.n, [&](int a, int b, int) {
        Numbering faces, cells;
        for (int k = a; k < b; k++) fill_tile(m, k, start[k + 1] - start[k], faces, cells, t);
    });
}

}  // namespace adfvm
