// CPU check of the order in which a tile's block tasks run (task_order,
// task_chunks): where the kernel has no shorter sum for the symmetric diagonal
// blocks, the chunks of 64 tasks hold the longest tasks first whatever their
// kind; where it has one, every chunk is of one kind and each kind is longest
// first.  T10 tiles: corner nodes have longer diagonal blocks than edge nodes,
// whose diagonal blocks are shorter than the corners' other ones.
// Prints "ok" and exits 0 when every check passes.
#include <algorithm>
#include <cstdio>
#include <set>
#include <vector>

#include "fused.hpp"

namespace feasm {
int64_t gen_t10block(double L, double W, double H, int64_t nL, int64_t nW, int64_t nH, double amp_v, double amp_m,
                     uint64_t seed, int64_t *conn10, std::vector<double> &xyz10);
// this program builds on the host only
std::shared_ptr<TileSet> build_tiles_device(feasm_mesh *, const TileShape &, hipStream_t) {
    throw Error(FEASM_EUNSUPPORTED, "no device in the tile check");
}
}  // namespace feasm

using namespace feasm;

static TileHostMesh t10(int n) {
    TileHostMesh h;
    h.npe = 10;
    h.ne = (int64_t)6 * n * n * n;
    std::vector<int64_t> c(h.ne * 10);
    h.nn = gen_t10block(1.0, 1.0, 1.0, n, n, n, 0.1 / n, 0.03 / n, 3, c.data(), h.xyz);
    h.n2e_ptr.assign(h.nn + 1, 0);
    for (int64_t v : c) {
        h.conn.push_back((int32_t)(v - 1));
        h.n2e_ptr[v]++;
    }
    for (int64_t i = 0; i < h.nn; i++) h.n2e_ptr[i + 1] += h.n2e_ptr[i];
    h.n2e.resize(h.ne * 10);
    std::vector<int64_t> cur(h.n2e_ptr.begin(), h.n2e_ptr.end() - 1);
    for (int64_t i = 0; i < h.ne * 10; i++) h.n2e[cur[h.conn[i]]++] = (uint32_t)(((i / 10) << 4) | (i % 10));
    h.adj_ptr.assign(1, 0);
    for (int64_t v = 0; v < h.nn; v++) {
        std::set<int32_t> l;
        for (int64_t s = h.n2e_ptr[v]; s < h.n2e_ptr[v + 1]; s++)
            for (int a = 0; a < 10; a++) l.insert(h.conn[(h.n2e[s] >> 4) * 10 + a]);
        h.adj.insert(h.adj.end(), l.begin(), l.end());
        h.adj_ptr.push_back((int64_t)h.adj.size());
    }
    return h;
}

struct Chunk {
    int first, last;
    bool sym, other;
};

static bool longest_first(std::vector<Chunk> c, const char *what, int64_t t) {
    std::sort(c.begin(), c.end(), [](const Chunk &a, const Chunk &b) {
        return a.first != b.first ? a.first > b.first : a.last > b.last;
    });
    for (size_t i = 1; i < c.size(); i++)
        if (c[i - 1].last < c[i].first) {
            std::fprintf(stderr, "%s, tile %lld: a chunk ends at %d items, a later one starts at %d\n", what,
                         (long long)t, c[i - 1].last, c[i].first);
            return false;
        }
    return true;
}

static bool check(const TileHostMesh &h, bool grad, const char *what) {
    TileShape s;
    s.npe = 10;
    s.nqp = 4;
    s.grad = grad;
    s.max_nodes = grad ? 64 : 32;
    s.threads = 1024;
    s.budget = 160 * 1024;
    HostTiles T;
    build_tiles_host(h, s, 2, T);
    for (int64_t t = 0; t < T.ntiles; t++) {
        const TileHdr &d = T.hdr[t];
        const TileShape::Layout L = s.layout(d.H, d.P, d.NH, d.K, d.NT, d.NI);
        const uint64_t *task = reinterpret_cast<const uint64_t *>(T.blob.get() + d.blob + (L.task - L.cbase));
        std::vector<Chunk> all, kind[2];
        for (int b = 0; b < d.NT; b += 64) {
            Chunk c{-1, -1, false, false};
            for (int i = b; i < std::min(d.NT, b + 64); i++) {
                const uint32_t w = (uint32_t)task[i];
                if (w == kNullTask) continue;
                const int k = (int)((w >> 16) & 255u);
                if (c.first < 0) c.first = k;
                if (c.last >= 0 && k > c.last && !(grad && c.sym && c.other)) {
                    std::fprintf(stderr, "%s, tile %lld: %d items after %d in a chunk\n", what, (long long)t, k, c.last);
                    return false;
                }
                c.last = k;
                ((w >> 26) & 1u ? c.sym : c.other) = true;
            }
            if (c.first < 0) continue;
            if (grad && c.sym && c.other) {
                std::fprintf(stderr, "%s, tile %lld: a chunk of both kinds\n", what, (long long)t);
                return false;
            }
            all.push_back(c);
            kind[c.sym].push_back(c);
        }
        if (grad ? !(longest_first(kind[0], what, t) && longest_first(kind[1], what, t)) : !longest_first(all, what, t))
            return false;
    }
    return true;
}

int main() {
    const TileHostMesh h = t10(5);
    if (!check(h, true, "gradient records") || !check(h, false, "dot")) return 1;
    std::printf("ok\n");
    return 0;
}
