// Which of a lane's forwards are worth a graph: the pairs of batch size and lanes in use that come often,
// whatever came first.
#pragma once
#include <cstdint>
#include <map>

namespace lzhip {

// Counts uses by key and holds the graphs of at most kMost keys.  A key gets one at its kAfter-th use; when
// all are taken, in the place of the least used one once it is used twice as often as that one (so that
// two sizes of about the same frequency do not take turns).  Every kAge uses the counts are halved, and
// what came long ago counts no more.  Graph: a pointer.
template <typename Graph>
class LayerGraphs {
public:
    static constexpr unsigned kAfter = 8, kMost = 16, kAge = 4096;

    // One more use of key: its graph, or null.  make() gives a graph, or null (then, and never for this
    // key again, plain launches it is); drop(graph) gives one up.
    template <typename Make, typename Drop>
    Graph use(int key, Make make, Drop drop) {
        if (++m_uses % kAge == 0) age();
        Entry& e = m_entries[key];
        e.uses++;
        if (e.graph || e.declined || e.uses < kAfter) return e.graph;
        if (m_graphs == kMost) {
            Entry* least = nullptr;
            for (auto& kv : m_entries)
                if (kv.second.graph && (!least || kv.second.uses < least->uses)) least = &kv.second;
            if (e.uses < 2 * least->uses) return nullptr;
            const Graph g = least->graph;
            least->graph = nullptr;
            m_graphs--;
            drop(g);
        }
        e.graph = make();
        if (e.graph) m_graphs++;
        else e.declined = true;
        return e.graph;
    }

    template <typename Drop>
    void clear(Drop drop) {
        for (auto& kv : m_entries)
            if (kv.second.graph) drop(kv.second.graph);
        m_entries.clear();
        m_graphs = 0;
    }

private:
    struct Entry {
        unsigned uses = 0;
        bool declined = false;
        Graph graph = nullptr;
    };
    void age() {
        for (auto it = m_entries.begin(); it != m_entries.end();) {
            it->second.uses /= 2;
            if (it->second.uses == 0 && !it->second.graph && !it->second.declined) it = m_entries.erase(it);
            else ++it;
        }
    }
    std::map<int, Entry> m_entries;
    unsigned m_graphs = 0;
    uint64_t m_uses = 0;
};

}  // namespace lzhip
