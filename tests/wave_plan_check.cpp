// Host check of the plans that deal a tile's ghost chunks to its waves
// (mr-lbm_amd/csrc/halo.h): every incoming chunk is moved by exactly one wave,
// the slots of one face window from the tile across the face by the same one;
// every outgoing chunk belongs to exactly one unit, whose chunks differ in
// their slot alone, as the kernel's one address and one set of terms per unit
// assume. Prints "ok" and exits 0 on success.
#include <cstdio>
#include <map>
#include <utility>
#include <vector>

#include "../mr-lbm_amd/csrc/halo.h"

using namespace mrlbm;

static int failures = 0;

#define CHECK(cond, ...)                              \
    do {                                              \
        if (!(cond)) {                                \
            failures++;                               \
            std::printf("Q%d %dx%dx%d: ", Q, BX, BY, BZ); \
            std::printf(__VA_ARGS__);                 \
            std::printf("\n");                        \
        }                                             \
    } while (0)

template <int Q, int BX, int BY, int BZ>
void check_shape() {
    using CT = ChunkTables<Q, BX, BY, BZ>;
    using IP = InPlan<Q, BX, BY, BZ>;
    constexpr auto plan = in_plan_v<Q, BX, BY, BZ>;
    std::vector<int> seen(CT::in.size(), 0);
    std::map<std::pair<int, int>, int> wave_of;  // face window -> wave of its direct chunks
    CHECK((int)CT::in.size() == IP::NIN, "%d chunks, plan for %d", (int)CT::in.size(), IP::NIN);
    for (int w = 0; w < IP::NW; w++) {
        CHECK(plan.n[w] >= 0 && plan.n[w] <= plan.rmax(), "wave %d holds %d of %d", w, plan.n[w], plan.rmax());
        for (int r = 0; r < plan.n[w]; r++) {
            const int k = plan.id[w][r];
            CHECK(k >= 0 && k < IP::NIN, "wave %d chunk %d", w, k);
            if (k < 0 || k >= IP::NIN) continue;
            seen[k]++;
            const Chunk& c = CT::in[k];
            if (IP::direct(c)) {
                const auto at = wave_of.emplace(std::make_pair(c.face, c.w0), w).first;
                CHECK(at->second == w, "face %d window %d in waves %d and %d", c.face, c.w0, at->second, w);
            }
        }
    }
    for (int k = 0; k < IP::NIN; k++) CHECK(seen[k] == 1, "incoming chunk %d moved %d times", k, seen[k]);

    using OU = OutUnits<Q, BX, BY, BZ>;
    constexpr int QF = VS<Q>::QF;
    std::vector<int> sent(CT::out.size(), 0);
    CHECK(OU::N * QF == (int)CT::out.size(), "%d units for %d chunks", OU::N, (int)CT::out.size());
    for (int u = 0; u < OU::N; u++) {
        const Chunk& a = CT::out[OU::chunk(u, 0)];
        for (int s = 0; s < QF; s++) {
            const int k = OU::chunk(u, s);
            CHECK(k >= 0 && k < (int)CT::out.size(), "unit %d slot %d: chunk %d", u, s, k);
            if (k < 0 || k >= (int)CT::out.size()) continue;
            sent[k]++;
            const Chunk& c = CT::out[k];
            CHECK(c.slot == s && c.pop == face_pop(a.face, s), "unit %d slot %d: slot %d pop %d", u, s, c.slot, c.pop);
            CHECK(c.face == a.face && c.w0 == a.w0 && c.rows == a.rows && c.ulo == a.ulo && c.uhi == a.uhi &&
                      c.vlo == a.vlo && c.vhi == a.vhi && c.lds0 == a.lds0 && c.su == a.su && c.sv == a.sv,
                  "unit %d slot %d differs from its first", u, s);
        }
    }
    for (size_t k = 0; k < sent.size(); k++) CHECK(sent[k] == 1, "outgoing chunk %d sent %d times", (int)k, sent[k]);
}

int main() {
#define SHAPE(A, B, C)          \
    check_shape<19, A, B, C>(); \
    check_shape<27, A, B, C>();
    SHAPE(8, 8, 8)
    SHAPE(16, 8, 4)
    SHAPE(32, 4, 4)
    SHAPE(64, 4, 2)
    SHAPE(16, 8, 8)
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
