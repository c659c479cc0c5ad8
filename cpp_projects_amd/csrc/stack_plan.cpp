// stack_plan.cpp -- groups and LDS layouts of the stacked merge passes.
#include "stack_plan.hpp"

#include <algorithm>
#include <stdexcept>

namespace sps {

namespace {

int32_t up4(int64_t v) { return (int32_t)((v + 3) & ~(int64_t)3); }  // (v >= 0)

// Windows of the rows of one state that a group reads: shifts lo..hi per row.
// (One record a row: a plan's build asks for some 70 windows per output row,
// and three arrays made that most of it.)
struct Windows {
    struct Row {
        int32_t lo, hi, stamp, pad;
    };
    std::vector<Row> row;
    std::vector<int32_t> rows;  // rows of the current group, in order of first use
    int32_t epoch = 0;
    void resize(size_t n) { row.assign(n, Row{0, 0, -1, 0}); }
    void clear() {
        ++epoch;
        rows.clear();
    }
    int32_t lo(int64_t r) const { return row[(size_t)r].lo; }
    int32_t hi(int64_t r) const { return row[(size_t)r].hi; }
};

// Tree of one row: leaf rows (-1: under a missing head) and their shifts, in
// heap-leaf order.
struct Tree {
    int32_t leaf[8];
    int32_t shift[8];
};

// The trees of the live rows of state `top` over state `bot`, at most three
// iterations below: a row's is its tail's followed by its head's, later by the
// offset.
std::vector<Tree> trees_of(const EnginePlan& eng, const std::vector<std::vector<uint8_t>>& live, int bot, int top) {
    std::vector<Tree> cur, prev;
    for (int i = bot; i <= top; ++i) {
        prev.swap(cur);
        const size_t n = (size_t)eng.rows[(size_t)i];
        cur.resize(n);
        if (i == bot) {
            for (size_t r = 0; r < n; ++r) {
                cur[r].leaf[0] = (int32_t)r;
                cur[r].shift[0] = 0;
            }
            continue;
        }
        const int half = 1 << (i - 1 - bot);
        for (size_t r = 0; r < n; ++r) {
            if (!live[(size_t)i][r]) continue;
            const RowDesc& rd = eng.iter[(size_t)i][r];
            const Tree& a = prev[(size_t)rd.tail_row];
            const bool head = rd.head_row >= 0;
            const Tree& b = prev[head ? (size_t)rd.head_row : (size_t)rd.tail_row];
            const int64_t off = head ? rd.offset : 0;
            Tree& t = cur[r];
            for (int k = 0; k < half; ++k) {
                t.leaf[k] = a.leaf[k];
                t.shift[k] = a.shift[k];
            }
            for (int k = 0; k < half; ++k) {
                const int64_t sh = b.shift[k] + off;
                const bool leaf = head && b.leaf[k] >= 0;
                if (leaf && sh > (int64_t)1 << 30) throw std::runtime_error("shift too large");
                t.leaf[half + k] = leaf ? b.leaf[k] : -1;
                t.shift[half + k] = leaf ? (int32_t)sh : 0;
            }
        }
    }
    return cur;
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
        tree_a = trees_of(eng, live, bot, mid);
        tree_b = trees_of(eng, live, mid, top);
        ub.resize(init ? (size_t)eng.nchans : (size_t)eng.rows[(size_t)bot]);
        rb.resize(init ? (size_t)eng.rows[0] : 0);
        ab.resize((size_t)eng.rows[(size_t)mid]);
    }

    StackTables run(bool weigh_init) {
        std::vector<int64_t> order;
        for (int64_t r = 0; r < eng.rows[(size_t)top]; ++r)
            if (live[(size_t)top][(size_t)r]) order.push_back(r);
        if (order.empty()) throw std::runtime_error("a pass without live rows");
        t.rows_a.reserve(order.size() + order.size() / 4 + kStackRowPad);
        t.rows_b.reserve(order.size() + kStackRowPad);
        t.tails.reserve(order.size() + order.size() / 4);
        const int64_t outputs = (int64_t)order.size() * kStackTile, tiles = (eng.nsamps + kStackTile - 1) / kStackTile;
        size_t q = 0, weighed = 0;
        int64_t steps = 0;  // of the groups so far, for one tile
        while (q < order.size()) {
            const size_t q0 = q;
            clear();
            while (q < order.size()) {
                nundo = 0;
                const int64_t f0 = floats_a, i0 = floats_i, u0 = units, t0 = tails;
                const size_t na = wa.rows.size(), nl = wl.rows.size(), nc = wc.rows.size();
                if (t.init) add_top<true>(order[q]);
                else add_top<false>(order[q]);
                if (fits()) {
                    ++q;
                    continue;
                }
                if (q == q0) throw std::runtime_error("one output row does not fit a stacked pass");
                while (nundo > 0) --nundo, *undo[nundo].row = undo[nundo].old;
                wa.rows.resize(na);
                wl.rows.resize(nl);
                wc.rows.resize(nc);
                floats_a = f0, floats_i = i0, units = u0, tails = t0;
                break;
            }
            emit(order, q0, q);
            if (!weigh_init) continue;
            for (; weighed < t.inits.size(); ++weighed) steps += (int64_t)t.inits[weighed].n * t.inits[weighed].k;
            if (steps > 2 * outputs && steps > ((int64_t)1 << 24) / tiles) return StackTables{};
        }
        t.rows_a.resize(t.rows_a.size() + kStackRowPad);
        t.rows_b.resize(t.rows_b.size() + kStackRowPad);
        return std::move(t);
    }

private:
    struct Undo {
        Windows::Row* row;
        Windows::Row old;
    };

    const EnginePlan& eng;
    const std::vector<std::vector<uint8_t>>& live;
    const int bot, top;
    int mid = 0;
    StackTables t;
    Windows wa, wl, wc;  // stage-A rows, leaf rows, channels (row 0, when init)
    std::vector<int32_t> row_chan;
    std::vector<Tree> tree_a, tree_b;
    Undo undo[8 + 2 * 64];  // an output row reads 8 stage-A rows, those 64 leaves (and their channels)
    int nundo = 0;
    int64_t floats_a = 0, floats_i = 0, units = 0, tails = 0;

    void clear() {
        wa.clear();
        wl.clear();
        wc.clear();
        floats_a = floats_i = units = tails = 0;
    }

    // Widens row r of w to shifts lo..hi; false when it held them already.
    // before: what it held (stamp: the epoch of w, unless this group had not
    // asked for it).
    static bool held(const Windows& w, const Windows::Row& x) { return x.stamp == w.epoch; }
    bool widen(Windows& w, int64_t r, int32_t lo, int32_t hi, Windows::Row& before) {
        Windows::Row& x = w.row[(size_t)r];
        before = x;
        const bool fresh = !held(w, x);
        if (!fresh && lo >= x.lo && hi <= x.hi) return false;
        undo[nundo++] = Undo{&x, x};
        if (fresh) {
            w.rows.push_back((int32_t)r);
            x = Windows::Row{lo, hi, w.epoch, 0};
        } else {
            x.lo = std::min(x.lo, lo);
            x.hi = std::max(x.hi, hi);
        }
        return true;
    }

    static int32_t unit_count(int32_t lo, int32_t hi) { return (kStackTile + up4(hi) - lo + 3) >> 2; }
    static int32_t tail_count(int32_t lo, int32_t hi) {
        return (int32_t)((uint32_t)(hi - lo + kStackTailLanes - 1) / kStackTailLanes);
    }

    void need_units(Windows& w, int64_t r, int32_t lo, int32_t hi) {
        Windows::Row b;
        if (widen(w, r, lo, hi, b)) units += unit_count(w.lo(r), w.hi(r)) - (held(w, b) ? unit_count(b.lo, b.hi) : 0);
    }

    template <bool INIT>
    void need_leaf(int64_t r, int32_t lo, int32_t hi) {
        if constexpr (!INIT) {
            need_units(wl, r, lo, hi);
        } else {
            // init row k of a channel: row 0 back to its k-th predecessor, and
            // its own window when k >= 1
            const int32_t c = row_chan[(size_t)r];
            const int32_t k = (int32_t)(r - eng.chan_row_off[(size_t)c]);
            need_units(wc, c, lo, hi + k);
            Windows::Row b;
            if (k > 0 && widen(wl, r, lo, hi, b))
                floats_i += wl.hi(r) - wl.lo(r) + (held(wl, b) ? b.lo - b.hi : kStackTile);
        }
    }

    template <bool INIT>
    void need_a(int64_t r, int32_t s) {
        Windows::Row b;
        if (!widen(wa, r, s, s, b)) return;
        const int32_t lo = wa.lo(r), hi = wa.hi(r);
        const bool had = held(wa, b);
        floats_a += hi - lo + (had ? b.lo - b.hi : kStackTile);
        tails += tail_count(lo, hi) - (had ? tail_count(b.lo, b.hi) : 0);
        const Tree& tr = tree_a[(size_t)r];
        for (int j = 0; j < (1 << t.la); ++j)
            if (tr.leaf[j] >= 0) need_leaf<INIT>(tr.leaf[j], lo + tr.shift[j], hi + tr.shift[j]);
    }

    template <bool INIT>
    void add_top(int64_t r) {
        const Tree& tr = tree_b[(size_t)r];
        for (int j = 0; j < (1 << t.lb); ++j)
            if (tr.leaf[j] >= 0) need_a<INIT>(tr.leaf[j], tr.shift[j]);
    }

    int64_t total_floats() const {
        return 4 * units + floats_i + floats_a + kStackTile + 4 + tails * (int64_t)(sizeof(StackTail) / 4);
    }

    bool fits() const {
        const size_t nl = t.init ? wc.rows.size() : wl.rows.size();
        return total_floats() <= kStackLdsFloats && units <= kStackMaxUnits && nl <= (size_t)kStackMaxLeaves &&
               (!t.init || nl <= (size_t)kStackMaxChans);
    }

    void emit(const std::vector<int64_t>& order, size_t q0, size_t q1) {
        StackGroup g{};
        int32_t off = 0;
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
            lf.smax4 = up4(wu.hi(r));
            g.smax4 = std::max(g.smax4, lf.smax4);
            lf.lds_off = off;
            lf.nunits = (int32_t)unit_count(wu.lo(r), wu.hi(r));
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
                const int32_t hi = wl.hi(r);
                StackInitRow ir{};
                ir.k = (int32_t)(r - eng.chan_row_off[(size_t)c]);
                ir.n = kStackTile + hi - wl.lo(r);
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
        for (int32_t r : wa.rows) a_off += kStackTile + wa.hi(r) - wa.lo(r);
        g.zero_off = a_off;
        g.tail_off = up4(a_off + kStackTile);
        g.tail0 = (int32_t)t.tails.size();
        for (int32_t r : wa.rows) {
            const int32_t lo = wa.lo(r), hi = wa.hi(r), span = hi - lo;
            // the window starts at time T - hi; its main samples at T - lo
            int32_t c[8];
            const Tree& tr = tree_a[(size_t)r];
            for (int j = 0; j < 8; ++j) {
                c[j] = g.zero_off;
                if (j < (1 << t.la) && tr.leaf[j] >= 0) {
                    c[j] = leaf_base(tr.leaf[j]) - tr.shift[j] - lo;
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
            const Tree& tr = tree_b[(size_t)order[q]];
            for (int j = 0; j < 8; ++j) {
                c[j] = g.zero_off;
                if (j < (1 << t.lb) && tr.leaf[j] >= 0) {
                    c[j] = a_base(tr.leaf[j]) - tr.shift[j];
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
    int32_t& unit_base(int64_t r) { return ub[(size_t)r]; }
    int32_t& row_base(int64_t r) { return rb[(size_t)r]; }
    int32_t& a_base(int64_t r) { return ab[(size_t)r]; }
    int32_t leaf_base(int64_t r) {
        if (!t.init) return unit_base(r);
        const int32_t c = row_chan[(size_t)r];
        return r == eng.chan_row_off[(size_t)c] ? unit_base(c) : row_base(r);
    }
};

}  // namespace

StackTables build_stack_pass(const EnginePlan& eng, const std::vector<std::vector<uint8_t>>& live, int i0, int depth,
                             bool init, bool weigh_init) {
    if (depth < 1 || depth > kStackMaxDepth || i0 < 1 || i0 + depth - 1 > eng.niters)
        throw std::invalid_argument("stacked pass out of the plan");
    if (init && i0 != 1) throw std::invalid_argument("only the first pass can build state 0");
    if (init && eng.nchans > (int64_t)1 << kStackChanBits) throw std::runtime_error("channels do not fit a slot");
    return Builder(eng, live, i0, depth, init).run(init && weigh_init);
}

int stack_threads(const StackTables& t) {
    int32_t rows = 0, units = 0, leaves = 0;
    for (const StackGroup& g : t.groups) {
        rows = std::max(rows, std::max(g.nrows_a, g.nrows_b));
        units = std::max(units, g.nunits);
        leaves = std::max(leaves, g.nleaves);
    }
    auto holds = [&](int threads) { return units <= threads * kStackSlots && leaves <= threads; };
    if (t.lds_floats > 8192) return kStackThreads;  // (small blocks gain by their number on a CU)
    if (rows <= 4 && holds(kStackFew4)) return kStackFew4;
    return rows <= 16 && holds(kStackFew16) ? kStackFew16 : kStackThreads;
}

}  // namespace sps
