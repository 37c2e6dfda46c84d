// Test shim: the cell tiles of adfvm_amd/csrc/tiles.hpp through C, compiled
// for the host with g++.
#include <cstring>

#include "tiles.hpp"

using namespace adfvm;

static Tiles t;

extern "C" int tiles_build(int nIC, int nIF, int nF, const int* sFace, const int* sOther, const int* sPair,
                           const unsigned char* sFlags, const unsigned char* fKind, unsigned copyBit) {
    t = Tiles();
    build_tiles(TileMesh{nIC, nIF, nF, sFace, sOther, sPair, sFlags, fKind, copyBit}, t);
    return t.n;
}

extern "C" void tiles_get(int* toUser, int* toTile, int* halo, int* faceId, unsigned* face, uint64_t* slots,
                          uint64_t* pairs, uint64_t* nbr) {
    auto put = [](auto* to, const auto& v) { std::memcpy(to, v.data(), v.size() * sizeof(v[0])); };
    put(toUser, t.toUser); put(toTile, t.toTile); put(halo, t.halo); put(faceId, t.faceId); put(face, t.face);
    put(slots, t.slots); put(pairs, t.pairs); put(nbr, t.nbr);
}
