// Runs of operations on tiny tensors (tiny.hip) as kernels of their own, compiled at run time.
//
// tiny.hip's kernels read a description of the run: finding a node's code and operands costs 0.5 us a node whatever it
// computes, and every node meets at a barrier and goes through LDS.  A plan runs the same run every time, so here its nodes
// become straight-line code: element i of an elementwise value stays in a register of thread i mod the workgroup's size,
// single elements are computed by every thread, and only what another thread reads goes through LDS, with a barrier where
// somebody reads what was written since the last one.  Every node computes the expressions of its stand-alone kernel in
// their order (see tiny.hip), so the values are the same bits.  Still one workgroup: bound by the latency of the run's
// dependent steps, not by any rate.
// Loss and gradient of the softmax regression, 26 operations on 1000 values: 30 us as two launches of tiny.hip's kernel, now 5; the
// loss of the 784-512-512-10 network, 13 on 2560 values, 18 -> 4.7; of VGG-16, 13 on 1280, 25 -> 5.
#include <algorithm>
#include <cstring>
#include <list>
#include <mutex>
#include <string>

#include "common.h"
#include "pw_ops.h"

namespace {

using namespace dopt;

struct Expr {
    int arity;
    const char *text;
};
const Expr kExprs[] = {
#define DOPT_PW_ROW(name, arity, f32, i32) {arity, #f32},
    DOPT_PW_OPS(DOPT_PW_ROW)
#undef DOPT_PW_ROW
};
constexpr int kExprCount = (int)(sizeof(kExprs) / sizeof(kExprs[0]));
constexpr int kMaxLds = 36864;   // floats; a CU has 40960

std::string num(long long v) { return std::to_string(v); }

// A value of the run: what a node makes, or a range of memory that the run reads.
struct Value {
    int slot = 0, offset = 0, n = 0;   // bytes; elements
    bool held = true;                  // in registers: element i in thread i mod T, a single one in all; else in LDS only
    bool shared = false;               // needs a place in LDS
    int at = -1;                       // that place
    int made = 0, last = -1;           // epochs (stretches between two barriers): written to LDS, last read there
};

struct Source {
    int value = -1;
    int skip = 0;   // elements into it
};

// How many values operand `which` of a node spans.
int extent(const dopt_hip_tiny_node &nd, int which)
{
    const int inner = nd.dims[0] > 0 ? nd.dims[0] : 1;
    switch (nd.kind) {
    case DOPT_HIP_TINY_POINTWISE: {
        const int kind = which == 0 ? nd.a_kind : nd.b_kind;
        return kind == 0 ? nd.n : kind == 1 ? 1 : kind == 2 ? nd.n / inner : inner;
    }
    case DOPT_HIP_TINY_REDUCE: return nd.dims[0] * nd.dims[1] * nd.dims[2];
    case DOPT_HIP_TINY_MATVEC: return which == 0 ? nd.n * nd.dims[0] : nd.dims[0];
    case DOPT_HIP_TINY_REPEAT: return nd.dims[0] * nd.dims[1] * nd.dims[2] * nd.dims[3];
    default: return nd.n;
    }
}

struct Generator {
    const std::vector<dopt_hip_tiny_node> &nodes;
    std::vector<Value> values;                 // the nodes' first, then what enters from outside
    std::vector<Source> from[2];               // per node: its operands
    int threads = 64, epoch = 0, lds = 0;
    bool emitting = false;
    std::string code;
    std::vector<int> unstored;                 // values in LDS that are not in memory yet

    explicit Generator(const std::vector<dopt_hip_tiny_node> &n) : nodes(n) {}

    bool binary(const dopt_hip_tiny_node &nd) const
    {
        return nd.kind == DOPT_HIP_TINY_SOFTMAX_GRAD || nd.kind == DOPT_HIP_TINY_MATVEC ||
               (nd.kind == DOPT_HIP_TINY_POINTWISE && kExprs[nd.op].arity == 2);
    }
    static bool row_fold(const dopt_hip_tiny_node &nd) { return nd.kind == DOPT_HIP_TINY_REDUCE && nd.dims[2] == 1 && nd.dims[1] > 64; }

    // Where every operand comes from: the latest earlier node whose result covers it, or memory.  False where ranges overlap in
    // part, or a node writes what another writes or the run reads from outside.
    bool resolve()
    {
        const int n = (int)nodes.size();
        for (int k = 0; k < n; k++) {
            const dopt_hip_tiny_node &nd = nodes[(size_t)k];
            if (nd.n < 1 || (nd.kind == DOPT_HIP_TINY_POINTWISE && (nd.op < 0 || nd.op >= kExprCount))) return false;
            Value v;
            v.slot = nd.dst;
            v.offset = nd.dst_offset;
            v.n = nd.n;
            // (a row's fold is known to all threads, many rows' folds to a thread each)
            v.held = !(nd.kind == DOPT_HIP_TINY_SOFTMAX || nd.kind == DOPT_HIP_TINY_SOFTMAX_GRAD || (row_fold(nd) && nd.dims[0] > 1) ||
                       (nd.kind == DOPT_HIP_TINY_MATVEC && nd.dims[0] > 16));
            v.shared = !v.held;
            values.push_back(v);
        }
        auto overlap = [](const Value &a, const Value &b) {
            return a.slot == b.slot && a.offset < b.offset + 4 * b.n && b.offset < a.offset + 4 * a.n;
        };
        for (int w = 0; w < 2; w++) from[w].assign((size_t)n, Source{});
        for (int k = 0; k < n; k++)
            for (int w = 0; w < (binary(nodes[(size_t)k]) ? 2 : 1); w++) {
                const dopt_hip_tiny_node &nd = nodes[(size_t)k];
                Value want;
                want.slot = w == 0 ? nd.a : nd.b;
                want.offset = w == 0 ? nd.a_offset : nd.b_offset;
                want.n = extent(nd, w);
                if (want.slot < 0 || want.n < 1) return false;
                Source &src = from[w][(size_t)k];
                for (int j = k - 1; j >= 0 && src.value < 0; j--) {
                    const Value &v = values[(size_t)j];
                    if (!overlap(v, want)) continue;
                    if (want.offset < v.offset || want.offset + 4 * want.n > v.offset + 4 * v.n) return false;
                    src = Source{j, (want.offset - v.offset) / 4};
                }
                for (size_t e = (size_t)n; e < values.size() && src.value < 0; e++)
                    if (values[e].slot == want.slot && values[e].offset == want.offset && values[e].n == want.n) src = Source{(int)e, 0};
                if (src.value < 0) {
                    values.push_back(want);
                    src = Source{(int)values.size() - 1, 0};
                }
                // read by another thread than the one that has it?
                Value &v = values[(size_t)src.value];
                const int kind = nd.kind == DOPT_HIP_TINY_POINTWISE ? (w == 0 ? nd.a_kind : nd.b_kind) : 1;
                const bool single = v.n == 1, own = nd.kind == DOPT_HIP_TINY_POINTWISE && kind == 0 && src.skip == 0 && v.n == nd.n;
                if (!single && !own) v.shared = true;
            }
        for (int j = 0; j < n; j++)
            for (size_t e = 0; e < values.size(); e++)
                if ((int)e != j && ((int)e > j || (int)e >= n) && overlap(values[(size_t)j], values[e])) return false;
        int most = 1;
        bool folds = false;
        for (const Value &v : values) most = std::max(most, v.n);
        for (const dopt_hip_tiny_node &nd : nodes) folds = folds || row_fold(nd) || (nd.kind == DOPT_HIP_TINY_MATVEC && nd.dims[0] > 16);
        threads = most > 512 ? 1024 : most > 256 ? 512 : most > 64 || folds ? 256 : 64;
        return true;
    }

    // ---- emission; run once to learn the epochs, once with the places in LDS known
    void put(const std::string &s)
    {
        if (emitting) code += s;
    }
    void barrier()
    {
        put("    __syncthreads();\n");
        epoch++;
        std::vector<int> keep;
        for (int v : unstored) {
            if (values[(size_t)v].made >= epoch) {
                keep.push_back(v);
                continue;
            }
            values[(size_t)v].last = epoch;
            for (int k = 0; k < passes(values[(size_t)v].n); k++) store(v, k, "L[" + num(values[(size_t)v].at) + " + " + index(values[(size_t)v].n, k) + "]");
        }
        unstored = keep;
    }
    int passes(int n) const { return (n + threads - 1) / threads; }
    // the element of pass k, kept inside the value
    std::string index(int n, int k) const
    {
        if (n == 1) return "0";
        const std::string i = k ? "(t + " + num((long long)k * threads) + ")" : "t";
        return (k + 1) * threads <= n ? i : "min(" + i + ", " + num(n - 1) + ")";
    }
    std::string inside(int n, int k) const
    {
        if (n == 1) return "if (t == 0) ";
        return (k + 1) * threads <= n ? "" : "if (t + " + num((long long)k * threads) + " < " + num(n) + ") ";
    }
    std::string name(int v, int k) const
    {
        const std::string s = (v < (int)nodes.size() ? "v" : "x") + num(v);
        return values[(size_t)v].n == 1 ? s : s + "_" + num(k);
    }
    std::string memory(int v) const { return "(p" + num(values[(size_t)v].slot) + " + " + num(values[(size_t)v].offset / 4) + ")"; }
    void store(int v, int k, const std::string &value)
    {
        put("    " + inside(values[(size_t)v].n, k) + memory(v) + "[" + (values[(size_t)v].n == 1 ? "0" : "t + " + num((long long)k * threads)) + "] = " + value + ";\n");
    }
    // a held value's places: LDS where another thread reads it, memory if a node made it
    void publish(int v)
    {
        Value &val = values[(size_t)v];
        for (int k = 0; k < passes(val.n); k++) {
            if (v < (int)nodes.size()) store(v, k, name(v, k));
            if (val.shared)
                put("    " + inside(val.n, k) + "L[" + num(val.at) + " + " + (val.n == 1 ? "0" : "t + " + num((long long)k * threads)) + "] = " + name(v, k) + ";\n");
        }
        val.made = epoch;
    }
    // before a node reads a value in LDS
    void meet(const Source &s, bool through_lds)
    {
        if (s.value >= 0 && through_lds && values[(size_t)s.value].made == epoch) barrier();
    }
    bool through_lds(const dopt_hip_tiny_node &nd, int w, const Source &s) const
    {
        const Value &v = values[(size_t)s.value];
        if (v.n == 1) return !v.held;
        const int kind = nd.kind == DOPT_HIP_TINY_POINTWISE ? (w == 0 ? nd.a_kind : nd.b_kind) : 1;
        return !(v.held && nd.kind == DOPT_HIP_TINY_POINTWISE && kind == 0 && s.skip == 0 && v.n == nd.n);
    }
    // element `i` (text) of an operand in LDS, or the held single value
    std::string at(const Source &s, const std::string &i)
    {
        Value &v = values[(size_t)s.value];
        if (v.n == 1 && v.held) return name(s.value, 0);
        v.last = epoch;
        return "L[" + num(v.at + s.skip) + " + " + i + "]";
    }

    void node(int k)
    {
        const dopt_hip_tiny_node &nd = nodes[(size_t)k];
        const Source a = from[0][(size_t)k], b = from[1][(size_t)k];
        meet(a, through_lds(nd, 0, a));
        if (b.value >= 0) meet(b, through_lds(nd, 1, b));
        Value &out = values[(size_t)k];
        const int n = nd.n;
        switch (nd.kind) {
        case DOPT_HIP_TINY_POINTWISE: {
            for (int q = 0; q < passes(n); q++) {
                auto operand = [&](const Source &s, int w, int kind) {
                    if (!through_lds(nd, w, s)) return name(s.value, q);
                    const std::string i = index(n, q), inner = num(nd.dims[0] > 0 ? nd.dims[0] : 1);
                    return at(s, kind == 0 ? i : kind == 1 ? "0" : kind == 2 ? "(" + i + ") / " + inner : "(" + i + ") % " + inner);
                };
                const std::string x = operand(a, 0, nd.a_kind), y = b.value >= 0 ? operand(b, 1, nd.b_kind) : x;
                put("    const float " + name(k, q) + " = f" + num(nd.op) + "(" + x + ", " + y + ");\n");
            }
            publish(k);
            break;
        }
        case DOPT_HIP_TINY_REDUCE: {
            const int outer = nd.dims[0], R = nd.dims[1], inner = nd.dims[2];
            const std::string f = nd.op == 0 ? "fold_sum" : "fold_max", ident = nd.op == 0 ? "0.0f" : "-3.402823466e+38f";
            if (!row_fold(nd)) {   // red_cols
                for (int q = 0; q < passes(n); q++) {
                    const std::string i = index(n, q), acc = name(k, q);
                    put("    float " + acc + " = " + ident + ";\n    {\n        const int o = (" + i + ") / " + num(inner) + ", j = (" + i + ") - o * " + num(inner) +
                        ";\n");
                    put("#pragma unroll 8\n        for (int r = 0; r < " + num(R) + "; r++) " + acc + " = " + f + "(" + acc + ", " +
                        at(a, "(o * " + num(R) + " + r) * " + num(inner) + " + j") + ");\n    }\n");
                }
                publish(k);
                break;
            }
            // red_rows / red_rows4: 256 threads a row, as many rows at a time as there are such groups
            const int groups = outer == 1 ? 1 : threads / 256;
            for (int o = 0; o < outer; o += groups) {
                const int now = std::min(groups, outer - o);
                const std::string part = "P[" + num(parts) + " + ";
                put("    if (t < " + num(256 * now) + ") {\n        const int u = t & 255, row = (" + num(o) + " + (t >> 8)) * " + num(R) + ";\n");
                put("        float a0 = " + ident + ", a1 = a0, a2 = a0, a3 = a0;\n        int i = u;\n");
                const bool quads = R % 4 == 0;
                const int steps = quads ? R / 4 : R;
                auto element = [&](const std::string &i) {
                    if (!quads) return at(a, "row + " + i);
                    auto e = [&](int c) { return at(a, "row + 4 * (" + i + ") + " + num(c)); };
                    return f + "(" + f + "(" + e(0) + ", " + e(1) + "), " + f + "(" + e(2) + ", " + e(3) + "))";
                };
                put("        for (; i + 768 < " + num(steps) + "; i += 1024) {\n");
                for (int c = 0; c < 4; c++) put("            a" + num(c) + " = " + f + "(a" + num(c) + ", " + element("i + " + num(256 * c)) + ");\n");
                put("        }\n        for (; i < " + num(steps) + "; i += 256) a0 = " + f + "(a0, " + element("i") + ");\n");
                put("        float v = " + f + "(" + f + "(a0, a1), " + f + "(a2, a3));\n#pragma unroll\n        for (int off = 32; off > 0; off >>= 1) v = " + f +
                    "(v, __shfl_down(v, off, 64));\n        if ((t & 63) == 0) " + part + "(t >> 6)] = v;\n    }\n");
                barrier();
                auto total = [&](const std::string &base) {
                    return f + "(" + f + "(" + f + "(" + part + base + "], " + part + base + " + 1]), " + part + base + " + 2]), " + part + base + " + 3])";
                };
                if (outer == 1) put("    const float " + name(k, 0) + " = " + total("0") + ";\n");
                else put("    if ((t & 255) == 0 && t < " + num(256 * now) + ") L[" + num(out.at + o) + " + (t >> 8)] = " + total("(t >> 6)") + ";\n");
                parts += 4 * now;
            }
            if (outer == 1) {
                publish(k);
            } else {
                out.made = epoch;
                unstored.push_back(k);
            }
            break;
        }
        case DOPT_HIP_TINY_SOFTMAX:
        case DOPT_HIP_TINY_SOFTMAX_GRAD: {
            const int C = nd.dims[1], inner = nd.dims[2], rows = nd.dims[0] * inner;
            const bool grad = nd.kind == DOPT_HIP_TINY_SOFTMAX_GRAD, few = C <= 32;
            for (int q = 0; q < passes(rows); q++) {
                const std::string i = index(rows, q), o = "L[" + num(out.at) + " + base + c * " + num(inner) + "]";
                const std::string x = at(a, "base + c * " + num(inner)), y = grad ? at(b, "base + c * " + num(inner)) : "", loop = "for (int c = 0; c < " + num(C) + "; c++) ";
                put("    " + (rows == 1 ? std::string("if (t == 0) ") : inside(rows, q)) + "{\n        const int i = " + i + ", base = i / " + num(inner) + " * " + num(C * inner) + " + i % " +
                    num(inner) + ";\n");
                if (few && !grad) {
                    const std::string each = "#pragma unroll\n        " + loop;
                    put("        float x[" + num(C) + "], m = -3.402823466e+38f, s = 0.0f;\n" + each + "x[c] = " + x + ";\n" + each + "m = m < x[c] ? x[c] : m;\n" + each +
                        "{ x[c] = expf(x[c] - m); s += x[c]; }\n" + each + o + " = x[c] / s;\n");
                } else if (!grad) {
                    put("        float m = -3.402823466e+38f, s = 0.0f;\n        " + loop + "{ const float v = " + x + "; m = m < v ? v : m; }\n        " + loop +
                        "{ const float pot = expf(" + x + " - m); s += pot; " + o + " = pot; }\n        " + loop + o + " = " + o + " / s;\n");
                } else if (few) {
                    const std::string each = "#pragma unroll\n        " + loop;
                    put("        float g[" + num(C) + "], y[" + num(C) + "], dot = 0.0f;\n" + each + "{ g[c] = " + x + "; y[c] = " + y + "; }\n" + each + "dot += g[c] * y[c];\n" +
                        each + o + " = y[c] * (g[c] - dot);\n");
                } else {
                    put("        float dot = 0.0f;\n        " + loop + "dot += " + x + " * " + y + ";\n        " + loop + o + " = " + y + " * (" + x + " - dot);\n");
                }
                put("    }\n");
            }
            out.made = epoch;
            unstored.push_back(k);
            break;
        }
        case DOPT_HIP_TINY_MATVEC: {
            const int K = nd.dims[0];
            if (K <= 16) {
                for (int q = 0; q < passes(n); q++) {
                    put("    float " + name(k, q) + ";\n    {\n        float q[16];\n        const int r = " + index(n, q) + " * " + num(K) + ";\n");
                    for (int c = 0; c < 16; c++)
                        put("        q[" + num(c) + "] = " + (c < K ? "0.0f + " + at(a, "r + " + num(c)) + " * " + at(b, num(c)) : std::string("0.0f")) + ";\n");
                    put("#pragma unroll\n        for (int c = 0; c < 16; c++) q[c] += 0.0f;\n#pragma unroll\n        for (int half = 8; half > 0; half /= 2)\n#pragma unroll\n"
                        "            for (int c = 0; c < half; c++) q[c] += q[c + half];\n        " + name(k, q) + " = q[0];\n    }\n");
                }
                publish(k);
                break;
            }
            put("    for (int r = t >> 6; r < " + num(n) + "; r += " + num(threads / 64) + ") {\n        float total = 0.0f;\n        for (int k0 = 0; k0 < " + num(K) +
                "; k0 += 1024) {\n            float acc = 0.0f;\n            for (int c = k0 + (t & 63); c < min(" + num(K) + ", k0 + 1024); c += 64) acc += " +
                at(a, "r * " + num(K) + " + c") + " * " + at(b, "c") + ";\n#pragma unroll\n            for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);\n" +
                "            total = k0 == 0 ? acc : total + acc;\n        }\n        if ((t & 63) == 0) L[" + num(out.at) + " + r] = total;\n    }\n");
            out.made = epoch;
            unstored.push_back(k);
            break;
        }
        default: {   // repeat
            const int o1 = nd.dims[1] * nd.reps[1], o2 = nd.dims[2] * nd.reps[2], o3 = nd.dims[3] * nd.reps[3];
            for (int q = 0; q < passes(n); q++) {
                const std::string i = "(" + index(n, q) + ")";
                const std::string c3 = i + " % " + num(o3), t3 = i + " / " + num(o3), c2 = t3 + " % " + num(o2), t2 = t3 + " / " + num(o2), c1 = t2 + " % " + num(o1),
                                  c0 = t2 + " / " + num(o1);
                const std::string src = "(((" + c0 + " % " + num(nd.dims[0]) + ") * " + num(nd.dims[1]) + " + " + c1 + " % " + num(nd.dims[1]) + ") * " + num(nd.dims[2]) + " + " +
                                        c2 + " % " + num(nd.dims[2]) + ") * " + num(nd.dims[3]) + " + " + c3 + " % " + num(nd.dims[3]);
                put("    const float " + name(k, q) + " = " + at(a, src) + ";\n");
            }
            publish(k);
        }
        }
    }
    int parts = 0;   // places of partial folds

    void pass()
    {
        epoch = parts = 0;
        unstored.clear();
        for (int e = (int)nodes.size(); e < (int)values.size(); e++)   // all loads together, then their places in LDS
            for (int k = 0; k < passes(values[(size_t)e].n); k++)
                put("    const float " + name(e, k) + " = " + memory(e) + "[" + index(values[(size_t)e].n, k) + "];\n");
        for (int e = (int)nodes.size(); e < (int)values.size(); e++) publish(e);
        for (int k = 0; k < (int)nodes.size(); k++) node(k);
        if (!unstored.empty()) barrier();
    }

    // Places in LDS: first fit among the values whose spans of epochs meet (one that was last read in an earlier epoch is gone).
    bool places()
    {
        struct Held { int at, len, last; };
        std::vector<Held> held;
        std::vector<int> order;
        for (int v = 0; v < (int)values.size(); v++)
            if (values[(size_t)v].shared) order.push_back(v);
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return values[(size_t)a].made < values[(size_t)b].made; });
        for (int v : order) {
            Value &val = values[(size_t)v];
            // (rows of a fold are written over several epochs, the first of them before `made`)
            const int first = v < (int)nodes.size() && row_fold(nodes[(size_t)v]) ? 0 : val.made, len = (val.n + 3) / 4 * 4;
            int at = 0;
            for (bool moved = true; moved;) {
                moved = false;
                for (const Held &h : held)
                    if (h.last >= first && at < h.at + h.len && h.at < at + len) {
                        at = h.at + h.len;
                        moved = true;
                    }
            }
            val.at = at;
            held.push_back({at, len, std::max(val.last, val.made)});
            lds = std::max(lds, at + len);
        }
        return lds + parts <= kMaxLds;
    }

    std::string source(int nslots)
    {
        std::string s = "__device__ inline float fold_sum(float a, float b) { return a + b; }\n"
                        "__device__ inline float fold_max(float a, float b) { return (a < b || a != a) ? b : a; }\ntypedef float T;\n";
        std::vector<char> have((size_t)kExprCount, 0);
        for (const dopt_hip_tiny_node &nd : nodes)
            if (nd.kind == DOPT_HIP_TINY_POINTWISE && !have[(size_t)nd.op]) {
                have[(size_t)nd.op] = 1;
                s += "__device__ inline float f" + num(nd.op) + "(float a, float b) { return (T)(" + kExprs[nd.op].text + "); }\n";
            }
        s += "extern \"C\" __global__ __launch_bounds__(" + num(threads) + ") void tiny_run(";
        for (int i = 0; i < nslots; i++) s += (i ? ", float *p" : "float *p") + num(i);
        s += ")\n{\n    __shared__ float L[" + num(std::max(4, lds)) + "], P[" + num(std::max(4, parts)) + "];\n    const int t = threadIdx.x;\n";
        return s + code + "}\n";
    }
};

}  // namespace

namespace dopt {

// The code objects of compiled runs, by their sources, the one that was asked for last at the back.  Runs with the same source
// share one.  Those that no run holds any more are kept for the next plan of the same network - compiling one takes 0.1 s - but
// only the kIdleCodes newest: a program that makes a plan for every batch size it meets would collect them.
struct TinyRun::Code {
    std::string source;
    hipModule_t module;
    hipFunction_t fn;   // null once the library has been shut down
};

namespace {

constexpr size_t kIdleCodes = 64;

struct Codes {
    std::mutex mutex;
    std::list<std::shared_ptr<TinyRun::Code>> all;
};
Codes &codes()
{
    static Codes *const c = new Codes;   // plans may be destroyed behind the end of main
    return *c;
}

// (mutex held)
void drop_idle(Codes &c, size_t keep)
{
    if (capturing()) return;   // nothing can be waited for now
    size_t idle = 0;
    for (const auto &code : c.all) idle += code.use_count() == 1;
    if (idle <= keep) return;
    rtc_idle();   // a kernel of a run that is gone may still be queued
    for (auto it = c.all.begin(); it != c.all.end() && idle > keep;) {
        if (it->use_count() != 1) {
            ++it;
            continue;
        }
        rtc_unload((*it)->module);
        it = c.all.erase(it);
        idle--;
    }
}

}  // namespace

void tiny_codes_trim()
{
    Codes &c = codes();
    std::lock_guard<std::mutex> lock(c.mutex);
    drop_idle(c, 0);
}

void tiny_codes_shutdown()
{
    Codes &c = codes();
    std::lock_guard<std::mutex> lock(c.mutex);
    for (const auto &code : c.all) {
        rtc_unload(code->module);
        code->fn = nullptr;
    }
    c.all.clear();
}

TinyRun::TinyRun(int nslots, const std::vector<dopt_hip_tiny_node> &nodes) : slots(nslots)
{
    Generator g(nodes);
    if (!g.resolve()) return;
    g.pass();
    if (!g.places()) return;
    g.emitting = true;
    g.pass();
    threads = g.threads;
    source = g.source(nslots);
}

TinyRun::~TinyRun()
{
    if (!code) return;
    Codes &c = codes();
    std::lock_guard<std::mutex> lock(c.mutex);
    code.reset();
    drop_idle(c, kIdleCodes);
}

// The run's kernel, compiled where no run with the same source has been.
int TinyRun::compile() const
{
    Codes &c = codes();
    std::lock_guard<std::mutex> lock(c.mutex);
    code.reset();
    for (auto it = c.all.begin(); it != c.all.end(); ++it)
        if ((*it)->source == source) {
            code = *it;
            c.all.splice(c.all.end(), c.all, it);
            return DOPT_HIP_OK;
        }
    auto made = std::make_shared<Code>();
    made->source = source;
    const char *const name = "tiny_run";
    if (int rc = rtc_load(source, 1, &name, &made->module, &made->fn)) return rc;
    c.all.push_back(made);
    code = made;
    drop_idle(c, kIdleCodes);
    return DOPT_HIP_OK;
}

int TinyRun::launch(void *const *ptrs, bool *done) const
{
    *done = false;
    if (threads == 0 || refused) return DOPT_HIP_OK;
    if (!code || !code->fn) {
        const std::string said = dopt_hip_last_error();
        if (compile()) {   // no compiler, no memory for the code: dopt_hip_tiny_graph needs neither
            refused = true;
            fail(DOPT_HIP_OK, "%s", said.c_str());   // what this call puts right is no error of its caller
            return DOPT_HIP_OK;
        }
    }
    void *args[DOPT_HIP_TINY_SLOTS];
    for (int i = 0; i < slots; i++) args[i] = (void *)&ptrs[i];
    *done = true;
    return rtc_launch(code->fn, 1, (unsigned)threads, args);
}

}  // namespace dopt
