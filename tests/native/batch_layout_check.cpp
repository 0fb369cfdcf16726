// The memory plan of batch runs (kunrt::batch_layout of libkunhip.so, host
// code) checked for built modules, over several sizes and lane counts:
//  * a node starts after every node that writes a buffer or handed-over value
//    it reads: the writer is an ancestor through the launch DAG's edges alone
//    (lane order is no substitute: an executor may spread lanes otherwise);
//  * values that share arena memory are never live together: every node
//    touching one of them precedes (through edges and lane order) the node
//    writing the other, and a value nothing writes shares with none;
//  * a plan for one lane needs no more memory than one for more lanes.
// Arguments: pairs of module name and library. Prints one line per violation
// and exits 1 if there was any.
#include <dlfcn.h>
#include <stdio.h>

#include <set>

#include "kun_rt.hpp"

using namespace kunrt;

static int bad = 0;

static void check(const KunModuleDesc *m, size_t S, size_t L, int lanes, const BatchLayout &lay) {
    const size_t N = lay.nodes.size();
    auto fail = [&](const char *what, size_t n, int a) {
        printf("%s %zu x %zu, %d lanes: node %zu (stage %d kernel %d): %s %d\n", m->name, S, L, lanes, n,
               lay.nodes[n].stage, lay.nodes[n].kern, what, a);
        bad++;
    };
    // ancestors by edges, and by edges and lane order
    std::vector<std::set<int>> by_dep(N), by_any(N);
    std::map<int, int> last;
    for (size_t n = 0; n < N; n++) {
        for (int d : lay.nodes[n].deps) {
            if (d < 0 || (size_t)d >= n) {
                fail("depends on a later node", n, d);
                continue;
            }
            by_dep[n].insert(d);
            by_dep[n].insert(by_dep[d].begin(), by_dep[d].end());
            by_any[n].insert(d);
            by_any[n].insert(by_any[d].begin(), by_any[d].end());
        }
        auto it = last.find(lay.nodes[n].lane);
        if (it != last.end()) {
            by_any[n].insert(it->second);
            by_any[n].insert(by_any[it->second].begin(), by_any[it->second].end());
        }
        last[lay.nodes[n].lane] = (int)n;
    }
    // values: module buffers, then every stage's handed-over values
    std::vector<int> first(m->nstage, 0);
    int nval = m->nbuf;
    for (int s = 0; s < m->nstage; s++) {
        first[s] = nval;
        if (m->stages[s].kind == KUN_STAGE_TS) nval += m->stages[s].nmat;
    }
    std::vector<int> writer(nval, -1);
    std::vector<std::vector<int>> reads(N), touch(nval);
    for (size_t n = 0; n < N; n++) {
        const KunStageDesc &sd = m->stages[lay.nodes[n].stage];
        std::vector<int> w;
        if (sd.kind == KUN_STAGE_TS) {
            const KunKernelDesc &kd = sd.kerns[lay.nodes[n].kern];
            reads[n].assign(kd.reads, kd.reads + kd.nreads);
            w.assign(kd.writes, kd.writes + kd.nwrites);
            for (int i = 0; i < kd.nmat_reads; i++) reads[n].push_back(first[lay.nodes[n].stage] + kd.mat_reads[i]);
            for (int i = 0; i < kd.nmat_writes; i++) w.push_back(first[lay.nodes[n].stage] + kd.mat_writes[i]);
        } else {
            reads[n].assign(sd.in, sd.in + sd.nin);
            w.assign(sd.out, sd.out + sd.nout);
        }
        for (int v : w) writer[v] = (int)n;
        for (int v : w) touch[v].push_back((int)n);
        for (int v : reads[n]) touch[v].push_back((int)n);
    }
    for (size_t n = 0; n < N; n++)
        for (int v : reads[n]) {
            if (v < m->nbuf && m->bufs[v].kind == KUN_BUF_INPUT) continue;
            if (writer[v] < 0) fail("reads a value nothing writes:", n, v);
            else if (writer[v] != (int)n && !by_dep[n].count(writer[v])) fail("does not wait for the writer of value", n, v);
        }
    std::map<size_t, std::vector<int>> at; // arena offset -> values there
    for (int b = 0; b < m->nbuf; b++)
        if (m->bufs[b].kind == KUN_BUF_TEMP) at[(size_t)lay.buf_off[b]].push_back(b);
    for (int s = 0; s < m->nstage; s++)
        for (size_t j = 0; j < lay.mat_off[s].size(); j++) at[lay.mat_off[s][j]].push_back(first[s] + (int)j);
    auto precedes = [&](int a, int b) { // every node touching a is done before b is written
        if (writer[a] < 0 || writer[b] < 0) return false;
        for (int t : touch[a])
            if (!by_any[writer[b]].count(t)) return false;
        return true;
    };
    for (auto &slot : at) {
        if (slot.first + lay.slot_bytes > lay.bytes) fail("slot past the arena's end, value", 0, slot.second[0]);
        auto nx = at.upper_bound(slot.first);
        if (nx != at.end() && nx->first < slot.first + lay.slot_bytes) fail("slots overlap, value", 0, slot.second[0]);
        for (size_t i = 0; i < slot.second.size(); i++)
            for (size_t j = 0; j < i; j++)
                if (!precedes(slot.second[i], slot.second[j]) && !precedes(slot.second[j], slot.second[i])) {
                    printf("%s %zu x %zu, %d lanes: values %d and %d live together in one slot\n", m->name, S, L, lanes,
                           slot.second[j], slot.second[i]);
                    bad++;
                }
    }
}

int main(int argc, char **argv) {
    const size_t sizes[][2] = {{64, 260}, {800, 500}, {8192, 1024}};
    int plans = 0;
    for (int i = 1; i + 1 < argc; i += 2) {
        void *h = dlopen(argv[i + 1], RTLD_NOW | RTLD_LOCAL);
        auto *m = h ? (const KunModuleDesc *)dlsym(h, (std::string("kun_module_") + argv[i]).c_str()) : nullptr;
        if (!m) {
            printf("cannot load %s from %s\n", argv[i], argv[i + 1]);
            return 1;
        }
        if (m->out_layout == KUN_LAYOUT_STREAM) continue;
        for (auto &sz : sizes) {
            const BatchLayout one = batch_layout(m, sz[0], sz[1], ChunkPolicy(), 1);
            check(m, sz[0], sz[1], 1, one);
            for (int lanes : {2, 4, 6}) {
                const BatchLayout lay = batch_layout(m, sz[0], sz[1], ChunkPolicy(), lanes);
                check(m, sz[0], sz[1], lanes, lay);
                if (one.bytes > lay.bytes) {
                    printf("%s %zu x %zu: %zu bytes on one lane, %zu on %d\n", m->name, sz[0], sz[1], one.bytes,
                           lay.bytes, lanes);
                    bad++;
                }
                plans++;
            }
        }
    }
    printf("%d plans\n", plans);
    return bad ? 1 : 0;
}
