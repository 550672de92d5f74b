// Host-only test of the table of layer graphs: which keys get one, and how many there are.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <stdexcept>

#include "layer_graphs.h"

#define CHECK(cond)                                                              \
    do {                                                                         \
        if (!(cond)) {                                                           \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #cond);              \
            std::exit(1);                                                        \
        }                                                                        \
    } while (0)

struct Table {
    typedef lzhip::LayerGraphs<int*> Graphs;
    Graphs graphs;
    std::set<int*> live;
    int made = 0;
    bool decline = false, fail = false;
    int* use(int key) {
        int* g = graphs.use(
            key,
            [&]() -> int* {
                if (fail) throw std::runtime_error("no graph");
                if (decline) return nullptr;
                made++;
                int* p = new int(key);
                live.insert(p);
                return p;
            },
            [&](int* p) { drop(p); });
        CHECK(live.size() <= Graphs::kMost);
        CHECK(!g || (live.count(g) && *g == key));
        return g;
    }
    void drop(int* p) {
        CHECK(live.erase(p) == 1);
        delete p;
    }
    void clear() {
        graphs.clear([&](int* p) { drop(p); });
        CHECK(live.empty());
    }
};

int main() {
    const int after = Table::Graphs::kAfter, most = Table::Graphs::kMost;
    {   // many sizes seen once or a few times leave room for the one that comes often
        Table t;
        for (int key = 1; key <= 200; key++)
            for (int i = 0; i < 1 + key % (after - 1); i++) CHECK(!t.use(key));
        for (int i = 1; i < after; i++) CHECK(!t.use(1000));
        for (int i = 0; i < 100; i++) CHECK(t.use(1000));
        CHECK(t.made == 1);
        t.clear();
        CHECK(!t.use(1000));
        t.clear();
    }
    {   // a full table: the frequent one comes in, equals do not take turns
        Table t;
        for (int i = 0; i < after; i++)
            for (int key = 0; key < 2 * most; key++) t.use(key);
        CHECK(t.made == most);
        for (int i = 0; i < 4 * after; i++) t.use(5000);
        CHECK(t.use(5000) && t.made == most + 1);
        for (int i = 0; i < 50; i++)
            for (int key = 0; key < 2 * most; key++) t.use(key);
        CHECK(t.made <= 2 * most + 1);
        t.clear();
    }
    {   // another phase of the program: sizes that were frequent make room
        Table t;
        for (int i = 0; i < 20000; i++) t.use(i % most);
        int first = 0;
        for (int i = 1; i <= 60000 && !first; i++)
            if (t.use(100 + i % most)) first = i;
        CHECK(first > 0 && first < 30000);
        for (int i = 0; i < 60000; i++) t.use(100 + i % most);
        for (int i = 0; i < most; i++) CHECK(t.use(100 + i));
        t.clear();
    }
    {   // what is declined is not asked for again; what fails leaves the table as it was
        Table t;
        t.decline = true;
        for (int i = 0; i < 100; i++) CHECK(!t.use(1));
        t.decline = false;
        CHECK(!t.use(1));
        t.fail = true;
        for (int i = 1; i < after; i++) CHECK(!t.use(2));
        for (int i = 0; i < 3; i++) {
            bool thrown = false;
            try {
                t.use(2);
            } catch (const std::runtime_error&) {
                thrown = true;
            }
            CHECK(thrown);
        }
        t.fail = false;
        CHECK(t.use(2));
        t.clear();
    }
    std::printf("layer graph tests passed\n");
    return 0;
}
