// The interpreter's form of a sweep program: the stack program's values numbered (equal operations
// on equal operands are one value, which they are bit for bit), its loads first, and the operations
// ordered into bundles of up to four independent ones of a kind.
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <unordered_map>
#include <vector>

#include "sweep.hpp"

namespace opf {

// Why bundles: a small sweep has about one wave per CU, so nothing hides a lane's own latencies.
// The stack program pays, instruction by instruction, the scalar load of the instruction, the LDS
// pop and, for a load, the memory: 0.2 to 0.3 us each. In this form the loads leave sixteen at a
// time, the next bundle is fetched while one runs, and a bundle pays its LDS latency and the
// dependent steps of its operation (a division: some 40 instructions) once for up to four.
constexpr int DAG_W = 4;
constexpr int DAG_LOADS = 16;      // loads in flight
// Values a lane keeps at a time (LDS); a program that needs more runs as a stack program. 96 hold
// every expression of the examples, at 48 KB a wave in FP64. The image ends with the stack program.
constexpr int DAG_MAX_SLOTS = 96;
constexpr int DAG_MAX_UNI = 96;    // constants (one copy a wave)

// operand and result words: a lane's value s as s << 1 | 1, constant c as c << 1
struct DagBundle {
    int op, sub;
    int d[DAG_W], a[DAG_W], b[DAG_W];  // I_SEL: condition a[0], b[0] where it holds, else a[1]
    int count, pad;                    // I_WENO_*: a[0..3], b[0..1] the values, b[2] the spacing
};
static_assert(sizeof(DagBundle) == 64, "one scalar load");
// src: 0 .. 7 a field, 8 + d the spacings and 11 + d the coordinates of dim d; ofs in elements
struct DagLoad {
    int src, ofs, d, pad;
};
// loads of a program in its image
inline __host__ __device__ int dag_loads(int n) { return (n + 7) / 8 * 8; }
struct DagUni {
    int slot, pad;  // launch-time constant, or -1: imm
    double imm;
};
struct DagBuilder {
    struct Node {
        int op, sub, ofs;  // loads: src and ofs; constants: launch slot and -1
        double imm;
        int a[7], na;
        int height = 0, uses = 0, slot = -1;
    };
    std::vector<Node> v;
    std::unordered_multimap<uint64_t, int> seen;

    int value(const Node& n) {
        uint64_t h = 1469598103934665603ull, bits;
        auto mix = [&](uint64_t x) { h = (h ^ x) * 1099511628211ull, h ^= h >> 29; };
        std::memcpy(&bits, &n.imm, 8);
        mix((uint64_t)(uint32_t)n.op << 32 | (uint32_t)n.sub), mix((uint32_t)n.ofs), mix(bits);
        for (int q = 0; q < n.na; ++q) mix((uint64_t)n.a[q]);
        for (auto r = seen.equal_range(h); r.first != r.second; ++r.first) {
            const Node& m = v[r.first->second];
            if (m.op == n.op && m.sub == n.sub && m.ofs == n.ofs && m.na == n.na &&
                std::memcmp(&m.imm, &n.imm, 8) == 0 && std::equal(n.a, n.a + n.na, m.a))
                return r.first->second;
        }
        seen.emplace(h, (int)v.size());
        v.push_back(n);
        return (int)v.size() - 1;
    }

    static int arity(int op) {
        switch (op) {
            case I_LD: case I_CONST: case I_DX: case I_X: return 0;
            case I_NEG: case I_ABS: case I_FN1: return 1;
            case I_SEL: return 3;
            case I_WENO_UP: case I_WENO_DOWN: return 7;
            case I_ADD: case I_SUB: case I_MUL: case I_DIV: case I_MIN: case I_MAX: case I_GT: case I_LT: case I_GE:
            case I_LE: case I_FN2: return 2;
            default: return -1;
        }
    }
    static int cost(int op) {
        switch (op) {
            case I_DIV: return 4;
            case I_FN1: case I_FN2: return 20;
            case I_WENO_UP: case I_WENO_DOWN: return 60;
            default: return 1;
        }
    }

    // false: more values alive at once than a lane has room for, or an operation that only the
    // stack program has
    bool build(const Insn* code, size_t n, std::vector<unsigned char>& out, DagInfo& info) {
        std::vector<int> st;
        for (size_t k = 0; k < n; ++k) {
            const Insn& in = code[k];
            Node x{};
            x.op = in.op;
            x.na = arity(in.op);
            if (x.na < 0 || (int)st.size() < x.na) return false;
            switch (in.op) {
                case I_LD: x.sub = in.a, x.ofs = in.b; break;
                case I_DX: x.sub = 8 + in.a, x.ofs = in.b; break;
                case I_X: x.sub = 11 + in.a, x.ofs = in.b; break;
                case I_CONST: x.sub = in.a ? in.b : -1, x.imm = in.a ? 0.0 : in.imm; break;
                case I_FN1: case I_FN2: x.sub = in.a; break;
                default: break;
            }
            if (in.op == I_DX || in.op == I_X) x.op = I_LD;
            for (int q = 0; q < x.na; ++q) x.a[q] = st[st.size() - x.na + q];
            st.resize(st.size() - x.na);
            st.push_back(value(x));
        }
        if (st.size() != 1) return false;
        const int root = st[0], nv = (int)v.size();
        // operands precede their values, so one backward pass gives heights and uses
        for (int k = nv - 1; k >= 0; --k)
            for (int q = 0; q < v[k].na; ++q) {
                Node& c = v[v[k].a[q]];
                ++c.uses;
                c.height = std::max(c.height, v[k].height + cost(v[k].op));
            }
        ++v[root].uses;
        std::vector<DagLoad> loads;
        std::vector<DagUni> unis;
        std::vector<int> word(nv, 0), free_slots;
        int nslot = 0;
        auto take = [&]() {
            if (free_slots.empty()) return nslot++;
            const int s = free_slots.back();
            free_slots.pop_back();
            return s;
        };
        std::vector<int> order;
        for (int k = 0; k < nv; ++k) {
            if (v[k].op == I_CONST) {
                word[k] = (int)unis.size() << 1;
                unis.push_back({v[k].sub, 0, v[k].imm});
            } else if (v[k].op == I_LD) {
                v[k].slot = take();
                word[k] = v[k].slot << 1 | 1;
                loads.push_back({v[k].sub, v[k].ofs, v[k].slot, 0});
            }
        }
        // operations by the longest way to the result; a bundle takes the first ready one and up to
        // three more of its kind
        std::vector<std::vector<int>> users(nv);
        std::vector<int> wait(nv, 0), ready;
        for (int k = 0; k < nv; ++k)
            for (int q = 0; q < v[k].na; ++q)
                if (v[v[k].a[q]].na > 0) users[v[k].a[q]].push_back(k), ++wait[k];
        auto before = [&](int x, int y) { return v[x].height != v[y].height ? v[x].height < v[y].height : x > y; };
        for (int k = 0; k < nv; ++k)
            if (v[k].na > 0 && wait[k] == 0) ready.push_back(k);
        std::sort(ready.begin(), ready.end(), before);
        std::vector<DagBundle> bundles;
        while (!ready.empty()) {
            const int op = v[ready.back()].op;
            const bool wide = op != I_SEL && op != I_WENO_UP && op != I_WENO_DOWN && op != I_FN1 && op != I_FN2;
            int pick[DAG_W], np = 0;
            for (int k = (int)ready.size() - 1; k >= 0 && np < (wide ? DAG_W : 1); --k)
                if (v[ready[k]].op == op) {
                    pick[np++] = ready[k];
                    ready.erase(ready.begin() + k);
                }
            DagBundle b{};
            b.op = op;
            b.sub = v[pick[0]].sub;
            b.count = np;
            for (int q = 0; q < np; ++q)
                for (int r = 0; r < v[pick[q]].na; ++r) {
                    const int w = word[v[pick[q]].a[r]];
                    if (op == I_SEL) (r == 0 ? b.a[0] : r == 1 ? b.b[0] : b.a[1]) = w;
                    else if (v[pick[q]].na == 7) (r < 4 ? b.a[r] : b.b[r - 4]) = w;
                    else (r == 0 ? b.a : b.b)[q] = w;
                }
            // every operand of a bundle is read before its results are written
            for (int q = 0; q < np; ++q)
                for (int r = 0; r < v[pick[q]].na; ++r) {
                    Node& c = v[v[pick[q]].a[r]];
                    if (--c.uses == 0 && c.slot >= 0) free_slots.push_back(c.slot);
                }
            for (int q = 0; q < np; ++q) {
                v[pick[q]].slot = take();
                word[pick[q]] = v[pick[q]].slot << 1 | 1;
                b.d[q] = word[pick[q]];
            }
            for (int q = np; q < DAG_W; ++q) {  // the spare places repeat the first operation
                b.d[q] = b.d[0];
                if (wide) b.a[q] = b.a[0], b.b[q] = b.b[0];
            }
            bundles.push_back(b);
            for (int q = 0; q < np; ++q)
                for (int u : users[pick[q]])
                    if (--wait[u] == 0) ready.insert(std::upper_bound(ready.begin(), ready.end(), u, before), u);
        }
        if (nslot > DAG_MAX_SLOTS || (int)unis.size() > DAG_MAX_UNI) return false;
        info.nload = (int)loads.size();
        info.nuni = (int)unis.size();
        info.nbundle = (int)bundles.size();
        info.nslot = std::max(nslot, 1);
        info.result = word[root];
        for (const DagBundle& b : bundles) info.cost += b.count > 1 ? 2 : 1;
        loads.resize(dag_loads(info.nload), loads.empty() ? DagLoad{} : loads[0]);  // a last group repeats one
        bundles.push_back(DagBundle{});  // read ahead of the last one
        out.clear();
        auto put = [&](const void* p, size_t bytes) {
            out.insert(out.end(), (const unsigned char*)p, (const unsigned char*)p + bytes);
        };
        put(bundles.data(), bundles.size() * sizeof(DagBundle));
        put(loads.data(), loads.size() * sizeof(DagLoad));
        put(unis.data(), unis.size() * sizeof(DagUni));
        info.stack = (int)out.size();
        put(code, n * sizeof(Insn));
        return true;
    }
};

}  // namespace opf
