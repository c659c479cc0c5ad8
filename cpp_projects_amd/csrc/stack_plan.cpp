// stack_plan.cpp -- groups and LDS layouts of the stacked merge passes.
#include "stack_plan.hpp"

#include <algorithm>
#include <stdexcept>

namespace sps {

namespace {

int32_t up4(int64_t v) { return (int32_t)((v + 3) / 4 * 4); }

// Windows of the rows of one state that a group reads: shifts lo..hi per row.
struct Windows {
    std::vector<int32_t> lo, hi, stamp;
    std::vector<int32_t> rows;  // rows of the current group, in order of first use
    int32_t epoch = 0;
    void resize(size_t n) {
        lo.assign(n, 0);
        hi.assign(n, 0);
        stamp.assign(n, -1);
    }
    void clear() {
        ++epoch;
        rows.clear();
    }
    bool has(int64_t r) const { return stamp[(size_t)r] == epoch; }
};

// Tree of one row, `L` iterations deep: leaf rows (-1: under a missing head)
// and their shifts, in heap-leaf order.
struct Tree {
    int64_t leaf[8];
    int64_t shift[8];
};

Tree tree_of(const EnginePlan& eng, int top, int L, int64_t row) {
    Tree t;
    int64_t node[16], sh[16];
    for (int k = 0; k < 16; ++k) node[k] = -1, sh[k] = 0;
    node[1] = row;
    int dep = 0;
    for (int k = 1; k < (1 << L); ++k) {
        while ((2 << dep) <= k) ++dep;
        if (node[k] < 0) continue;
        const RowDesc& rd = eng.iter[(size_t)(top - dep)][(size_t)node[k]];
        node[2 * k] = rd.tail_row;
        sh[2 * k] = sh[k];
        if (rd.head_row >= 0) {
            node[2 * k + 1] = rd.head_row;
            sh[2 * k + 1] = sh[k] + rd.offset;
        }
    }
    for (int j = 0; j < 8; ++j) {
        t.leaf[j] = j < (1 << L) ? node[(1 << L) + j] : -1;
        t.shift[j] = j < (1 << L) ? sh[(1 << L) + j] : 0;
    }
    return t;
}

class Builder {
public:
    Builder(const EnginePlan& e, const std::vector<std::vector<uint8_t>>& live, int i0, int depth, bool init)
        : eng(e), live(live), bot(i0 - 1), top(i0 + depth - 1) {
        t.init = init;
        // depth 6: 3 + 3, 5: 3 + 2, 4: 2 + 2, 3: 2 + 1, 2: 1 + 1, 1: 1 + 0 (stage B copies)
        t.la = (depth + 1) / 2;
        t.lb = depth - t.la;
        mid = bot + t.la;
        wa.resize((size_t)eng.rows[(size_t)mid]);
        wl.resize((size_t)eng.rows[(size_t)bot]);
        if (init) {
            wc.resize((size_t)eng.nchans);
            row_chan.resize((size_t)eng.rows[0]);
            for (int64_t c = 0; c < eng.nchans; ++c)
                for (int64_t q = eng.chan_row_off[(size_t)c]; q < eng.chan_row_off[(size_t)c + 1]; ++q)
                    row_chan[(size_t)q] = (int32_t)c;
        }
        {
            tree_a.resize((size_t)eng.rows[(size_t)mid]);
            for (int64_t r = 0; r < eng.rows[(size_t)mid]; ++r)
                if (live[(size_t)mid][(size_t)r]) tree_a[(size_t)r] = tree_of(eng, mid, t.la, r);
        }
    }

    StackTables run() {
        std::vector<int64_t> order;
        for (int64_t r = 0; r < eng.rows[(size_t)top]; ++r)
            if (live[(size_t)top][(size_t)r]) order.push_back(r);
        if (order.empty()) throw std::runtime_error("a pass without live rows");
        size_t q = 0;
        while (q < order.size()) {
            const size_t q0 = q;
            clear();
            while (q < order.size()) {
                undo.clear();
                const int64_t f0 = floats_a, l0 = floats_l, u0 = units, t0 = tails;
                const size_t na = wa.rows.size(), nl = wl.rows.size(), nc = wc.rows.size();
                add_top(order[q]);
                if (fits()) {
                    ++q;
                    continue;
                }
                if (q == q0) throw std::runtime_error("one output row does not fit a stacked pass");
                for (size_t k = undo.size(); k-- > 0;) {
                    const Undo& u = undo[k];
                    u.w->lo[(size_t)u.row] = u.lo;
                    u.w->hi[(size_t)u.row] = u.hi;
                    u.w->stamp[(size_t)u.row] = u.stamp;
                }
                wa.rows.resize(na);
                wl.rows.resize(nl);
                wc.rows.resize(nc);
                floats_a = f0, floats_l = l0, units = u0, tails = t0;
                break;
            }
            emit(order, q0, q);
        }
        t.rows_a.resize(t.rows_a.size() + kStackRowPad);
        t.rows_b.resize(t.rows_b.size() + kStackRowPad);
        return std::move(t);
    }

private:
    struct Undo {
        Windows* w;
        int64_t row;
        int32_t lo, hi, stamp;
    };

    const EnginePlan& eng;
    const std::vector<std::vector<uint8_t>>& live;
    const int bot, top;
    int mid = 0;
    StackTables t;
    Windows wa, wl, wc;  // stage-A rows, leaf rows, channels (row 0, when init)
    std::vector<int32_t> row_chan;
    std::vector<Tree> tree_a;
    std::vector<Undo> undo;
    int64_t floats_a = 0, floats_l = 0, units = 0, tails = 0;

    void clear() {
        wa.clear();
        wl.clear();
        wc.clear();
        floats_a = floats_l = units = tails = 0;
    }

    // widens row r of w to shifts lo..hi; false when it held them already
    bool widen(Windows& w, int64_t r, int32_t lo, int32_t hi, int32_t& olo, int32_t& ohi, bool& fresh) {
        fresh = !w.has(r);
        olo = w.lo[(size_t)r];
        ohi = w.hi[(size_t)r];
        if (!fresh && lo >= olo && hi <= ohi) return false;
        undo.push_back(Undo{&w, r, olo, ohi, w.stamp[(size_t)r]});
        if (fresh) {
            w.rows.push_back((int32_t)r);
            w.stamp[(size_t)r] = w.epoch;
            w.lo[(size_t)r] = lo;
            w.hi[(size_t)r] = hi;
        } else {
            w.lo[(size_t)r] = std::min(olo, lo);
            w.hi[(size_t)r] = std::max(ohi, hi);
        }
        return true;
    }

    static int64_t unit_count(int32_t lo, int32_t hi) { return (kStackTile + up4(hi) - lo + 3) / 4; }
    static int64_t tail_count(int32_t lo, int32_t hi) { return (hi - lo + kStackTailLanes - 1) / kStackTailLanes; }

    void need_units(Windows& w, int64_t r, int32_t lo, int32_t hi) {
        int32_t olo, ohi;
        bool fresh;
        if (!widen(w, r, lo, hi, olo, ohi, fresh)) return;
        const int64_t d = unit_count(w.lo[(size_t)r], w.hi[(size_t)r]) - (fresh ? 0 : unit_count(olo, ohi));
        units += d;
        floats_l += 4 * d;
    }

    void need_leaf(int64_t r, int32_t lo, int32_t hi) {
        if (!t.init) {
            need_units(wl, r, lo, hi);
            return;
        }
        // init row k of a channel: row 0 back to its k-th predecessor, and its
        // own window when k >= 1
        const int32_t c = row_chan[(size_t)r];
        const int32_t k = (int32_t)(r - eng.chan_row_off[(size_t)c]);
        need_units(wc, c, lo, hi + k);
        if (k == 0) return;
        int32_t olo, ohi;
        bool fresh;
        if (!widen(wl, r, lo, hi, olo, ohi, fresh)) return;
        floats_l += (wl.hi[(size_t)r] - wl.lo[(size_t)r] + (fresh ? kStackTile : 0)) - (fresh ? 0 : ohi - olo);
    }

    void need_a(int64_t r, int32_t s) {
        int32_t olo, ohi;
        bool fresh;
        if (!widen(wa, r, s, s, olo, ohi, fresh)) return;
        const int32_t lo = wa.lo[(size_t)r], hi = wa.hi[(size_t)r];
        floats_a += (hi - lo + (fresh ? kStackTile : 0)) - (fresh ? 0 : ohi - olo);
        tails += tail_count(lo, hi) - (fresh ? 0 : tail_count(olo, ohi));
        const Tree& tr = tree_a[(size_t)r];
        for (int j = 0; j < (1 << t.la); ++j)
            if (tr.leaf[j] >= 0) need_leaf(tr.leaf[j], lo + (int32_t)tr.shift[j], hi + (int32_t)tr.shift[j]);
    }

    void add_top(int64_t r) {
        const Tree tr = tree_of(eng, top, t.lb, r);
        for (int j = 0; j < (1 << t.lb); ++j)
            if (tr.leaf[j] >= 0) {
                if (tr.shift[j] > (int64_t)1 << 30) throw std::runtime_error("shift too large");
                need_a(tr.leaf[j], (int32_t)tr.shift[j]);
            }
    }

    int64_t total_floats() const {
        return floats_l + floats_a + kStackTile + 4 + tails * (int64_t)(sizeof(StackTail) / 4);
    }

    bool fits() const {
        const size_t nl = t.init ? wc.rows.size() : wl.rows.size();
        return total_floats() <= kStackLdsFloats && units <= kStackMaxUnits && nl <= (size_t)kStackMaxLeaves &&
               (!t.init || nl <= (size_t)kStackMaxChans);
    }

    void emit(const std::vector<int64_t>& order, size_t q0, size_t q1) {
        StackGroup g{};
        int32_t off = 0;
        std::vector<int32_t> base_l;  // per leaf row: float offset of time T
        Windows& wu = t.init ? wc : wl;
        std::sort(wu.rows.begin(), wu.rows.end());
        if (t.init) std::sort(wl.rows.begin(), wl.rows.end());
        std::sort(wa.rows.begin(), wa.rows.end());
        g.leaf0 = (int32_t)t.leaves.size();
        g.nleaves = (int32_t)wu.rows.size();
        g.unit0 = (int64_t)t.unit_leaf.size();
        int32_t u0 = 0;
        for (size_t k = 0; k < wu.rows.size(); ++k) {
            const int32_t r = wu.rows[k];
            StackLeaf lf{};
            lf.row = r;
            lf.smax4 = up4(wu.hi[(size_t)r]);
            g.smax4 = std::max(g.smax4, lf.smax4);
            lf.lds_off = off;
            lf.nunits = (int32_t)unit_count(wu.lo[(size_t)r], wu.hi[(size_t)r]);
            lf.unit0 = u0;
            u0 += lf.nunits;
            unit_base(r) = off + lf.smax4;
            off += 4 * lf.nunits;
            t.leaves.push_back(lf);
            t.unit_leaf.insert(t.unit_leaf.end(), (size_t)lf.nunits, (uint8_t)k);
        }
        g.nunits = u0;
        g.init0 = (int32_t)t.inits.size();
        if (t.init) {
            for (int32_t r : wl.rows) {
                const int32_t c = row_chan[(size_t)r];
                const int32_t hi = wl.hi[(size_t)r];
                StackInitRow ir{};
                ir.k = (int32_t)(r - eng.chan_row_off[(size_t)c]);
                ir.n = kStackTile + hi - wl.lo[(size_t)r];
                ir.t_off = hi;
                ir.c = unit_base(c) - hi;
                ir.out = off;
                row_base(r) = off + hi;
                off += ir.n;
                t.inits.push_back(ir);
            }
            g.ninit = (int32_t)wl.rows.size();
        }
        const int32_t leaf_end = off;
        g.row_a0 = (int32_t)t.rows_a.size();
        g.nrows_a = (int32_t)wa.rows.size();
        int32_t a_off = off;
        for (int32_t r : wa.rows) a_off += kStackTile + wa.hi[(size_t)r] - wa.lo[(size_t)r];
        g.zero_off = a_off;
        g.tail_off = up4(a_off + kStackTile);
        g.tail0 = (int32_t)t.tails.size();
        for (int32_t r : wa.rows) {
            const int32_t lo = wa.lo[(size_t)r], hi = wa.hi[(size_t)r], span = hi - lo;
            // the window starts at time T - hi; its main samples at T - lo
            int32_t c[8];
            const Tree& tr = tree_a[(size_t)r];
            for (int j = 0; j < 8; ++j) {
                c[j] = g.zero_off;
                if (j < (1 << t.la) && tr.leaf[j] >= 0) {
                    c[j] = leaf_base(tr.leaf[j]) - (int32_t)tr.shift[j] - lo;
                    check(c[j] - span >= 0 && c[j] + kStackTile <= leaf_end);
                }
            }
            for (int32_t s = 0; s < span; s += kStackTailLanes) {
                StackTail tl{};
                for (int j = 0; j < 8; ++j)
                    tl.c[j] = 4 * (c[j] == g.zero_off ? g.zero_off : c[j] - span + s);
                tl.out = 4 * (off + s);
                tl.n = std::min(kStackTailLanes, span - s);
                t.tails.push_back(tl);
            }
            t.rows_a.push_back(pack(c, t.la, 4 * (off + span)));
            a_base(r) = off + hi;
            off += kStackTile + span;
        }
        g.ntails = (int32_t)t.tails.size() - g.tail0;
        const int32_t end = g.tail_off + g.ntails * (int32_t)(sizeof(StackTail) / 4);
        check(off == a_off && end <= kStackLdsFloats);
        g.row_b0 = (int32_t)t.rows_b.size();
        g.nrows_b = (int32_t)(q1 - q0);
        for (size_t q = q0; q < q1; ++q) {
            int32_t c[8];
            const Tree tr = tree_of(eng, top, t.lb, order[q]);
            for (int j = 0; j < 8; ++j) {
                c[j] = g.zero_off;
                if (j < (1 << t.lb) && tr.leaf[j] >= 0) {
                    c[j] = a_base(tr.leaf[j]) - (int32_t)tr.shift[j];
                    check(c[j] >= leaf_end && c[j] + kStackTile <= a_off);
                }
            }
            check(order[q] <= INT32_MAX);
            t.rows_b.push_back(pack(c, t.lb, (int32_t)order[q]));
        }
        t.groups.push_back(g);
        t.lds_floats = std::max(t.lds_floats, end);
    }

    static StackRow pack(const int32_t (&c)[8], int L, int32_t out) {
        StackRow r{};
        for (int j = 0; j < (1 << L); ++j) {
            check(c[j] >= 0 && c[j] < (1 << 16));
            if (L <= 2) r.w[j] = 4u * (uint32_t)c[j];
            else r.w[j / 2] |= (uint32_t)c[j] << (16 * (j % 2));
        }
        r.out = out;
        return r;
    }
    static void check(bool ok) {
        if (!ok) throw std::runtime_error("stacked pass layout out of its windows");
    }

    // float offsets of time T in the windows (valid within emit)
    std::vector<int32_t> ub, rb, ab;
    int32_t& at(std::vector<int32_t>& v, int64_t r, size_t n) {
        if (v.size() < n) v.resize(n);
        return v[(size_t)r];
    }
    int32_t& unit_base(int64_t r) { return at(ub, r, t.init ? (size_t)eng.nchans : (size_t)eng.rows[(size_t)bot]); }
    int32_t& row_base(int64_t r) { return at(rb, r, (size_t)eng.rows[(size_t)bot]); }
    int32_t& a_base(int64_t r) { return at(ab, r, (size_t)eng.rows[(size_t)mid]); }
    int32_t leaf_base(int64_t r) {
        if (!t.init) return unit_base(r);
        const int32_t c = row_chan[(size_t)r];
        return r == eng.chan_row_off[(size_t)c] ? unit_base(c) : row_base(r);
    }
};

}  // namespace

StackTables build_stack_pass(const EnginePlan& eng, const std::vector<std::vector<uint8_t>>& live, int i0, int depth,
                             bool init) {
    if (depth < 1 || depth > kStackMaxDepth || i0 < 1 || i0 + depth - 1 > eng.niters)
        throw std::invalid_argument("stacked pass out of the plan");
    if (init && i0 != 1) throw std::invalid_argument("only the first pass can build state 0");
    if (init && eng.nchans > (int64_t)1 << kStackChanBits) throw std::runtime_error("channels do not fit a slot");
    return Builder(eng, live, i0, depth, init).run();
}

bool separate_init_faster(const StackTables& t, int64_t nsamps) {
    if (!t.init) return false;
    int64_t steps = 0, outputs = 0;  // of a tile
    for (const StackInitRow& r : t.inits) steps += (int64_t)r.n * r.k;
    for (const StackGroup& g : t.groups) outputs += (int64_t)g.nrows_b * kStackTile;
    return steps > 2 * outputs && steps * ((nsamps + kStackTile - 1) / kStackTile) > (int64_t)1 << 24;
}

}  // namespace sps
