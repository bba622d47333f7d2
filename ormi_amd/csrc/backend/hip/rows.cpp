// Row programs: reductions over the same trailing dims and the element-wise
// values around them, realized by one kernel that reads each operand once.
//
// A softmax, a normalization or the statistics of one tensor are several
// reductions over the rows of one shape S (its last k dims) and element-wise
// values over S, over its rows, or both. Realized one by one, each reduction
// and each map passes over the operands again; a row program keeps the row in
// registers from one stage to the next (plan_rows). The reference realizes
// every node on its own (csrc/backend/runtime.cpp:16-18).
//
// A program is built from its roots down. Its nodes have one of these forms:
//   full    shape S
//   keep    one value per row, shape S with the last k dims 1
//   kept    one value per row, shape S without the last k dims
//   scalar  one element
// A full node reads full, keep and scalar nodes (EXPAND from keep to S, and
// RESHAPE between keep and kept, only rename a value); keep reads keep and
// scalar, kept reads kept and scalar; a SUM or MAX of a full node over the
// last k dims is keep or kept. Whatever else a node reads is a leaf, realized
// first. Besides the roots the program stores every reduction it computes and
// every per-row value that a full node reads, so that what reads them later
// finds buffers.
#include <algorithm>
#include <vector>

#include "backend/hip/hip_backend.h"
#include "backend/hip/small_containers.h"
#include "core/memory.h"
#include "runtime/runtime.h"

namespace ormi::hip {
    using ops::OpEnum;

    namespace {
        constexpr int kMaxItems = 96;     // nodes of one program
        // Nodes one root may add, views that only rename a value included. An item
        // is added after its operands, so this, not kMaxItems, bounds how deep
        // a walk recurses and how much of a long chain a declined root reads.
        constexpr int kMaxVisits = 4 * kMaxItems;
        constexpr int kMaxReductions = 12;
        constexpr int kMaxHeld = 8;       // operands that vary along a row
        constexpr size_t kMaxColumns = 4;

        // The rows of shape `s`: its last k dims reduced.
        struct Space {
            std::vector<int> s;
            int k = 0;
            long long O = 1, R = 1;
        };
        bool make_space(const std::vector<int>& s, int k, Space* sp) {
            const int nd = (int)s.size();
            if (k < 1 || k >= nd) return false;
            sp->s = s;
            sp->k = k;
            sp->O = sp->R = 1;
            for (int d = 0; d < nd; ++d) (d < nd - k ? sp->O : sp->R) *= s[d];
            return sp->O >= 2 && sp->R >= 2;
        }
        // Dims a reduction removes, when they are the last ones (or, leading,
        // the first ones) of its input: their count, else 0.
        int trailing_axes(const Node& n, bool leading = false) {
            const auto& ax = std::get<ReduceAttrs>(n.attrs).axes;  // sorted
            const int nd = (int)n.parents[0]->view.shape.size(), m = (int)ax.size();
            if (m == 0 || m >= nd) return 0;
            for (int i = 0; i < m; ++i)
                if (ax[i] != (leading ? i : nd - m + i)) return 0;
            return m;
        }

        enum Form : char { Full, Keep, Kept, Scalar, None };

        struct Item {
            NodePtr n;
            Form form = None;
            bool leaf = false;
            bool kept_ctx = false;  // leaf aligned to the kept shape
            int a = -1, b = -1;
            bool boundary = false;  // a per-row op that a full node reads
        };

        class Builder {
        public:
            Space sp;
            std::vector<Item> items;       // operands before their readers
            std::vector<NodePtr> frontier;  // unrealized leaves
            struct Root {
                NodePtr n;
                int item;
                bool column;
            };
            std::vector<Root> roots;
            int reductions = 0, fulls = 0, columns = 0;

            Builder(const Space& s, bool plan_only = false) : sp(s), plan_only_(plan_only) {
                const int nd = (int)s.s.size();
                keep_ = s.s;
                for (int d = nd - s.k; d < nd; ++d) keep_[d] = 1;
                kept_.assign(s.s.begin(), s.s.end() - s.k);
                items.reserve(32);
            }

            // Adds root (a node of the program's space); false, with the
            // program's items as they were, when it does not belong to it: not of its
            // forms, no operand in common with what is there, too large, or a
            // reader of an ARGMAX that is there.
            bool add(const NodePtr& root) {
                const size_t ni = items.size(), nf = frontier.size();
                const int nr = reductions;
                over_ = touched_ = false;
                visits_ = 0;
                int it = -1;
                bool column = false;
                if (root->op == OpEnum::SUM && root->parents[0]->view.shape == sp.s && is_column(*root)) {
                    column = columns < (int)kMaxColumns;
                    if (column) it = visit(root->parents[0], Full);
                } else if (root->op == OpEnum::ARGMAX) {
                    if (is_row_reduction(*root)) it = reduce(root, form_any(root->view.shape));
                } else if (is_row_reduction(*root) || fusible_interior(*root)) {
                    const Form f = form_any(root->view.shape);
                    if (f != None && f != Scalar) it = visit(root, f);
                }
                const bool ok = it >= 0 && !over_ && (column || !items[it].leaf) && (roots.empty() || touched_) && held() <= kMaxHeld;
                if (!ok) {
                    // Boundary marks stay: the caller realizes root next, and it
                    // reads the values that they make the program store.
                    items.resize(ni);
                    frontier.resize(nf);
                    reductions = nr;
                    reindex();
                    return false;
                }
                roots.push_back({root, it, column});
                columns += column;
                fulls += !column && items[it].form == Full;
                return true;
            }

            // More than one pass over the operands saved.
            bool worthwhile() const { return reductions + columns >= 1 && reductions + fulls + columns >= 2; }

        private:
            std::vector<int> keep_, kept_;
            // Items by node, per context (right-aligned to S, or to the kept
            // shape): at most kMaxItems and their views, searched linearly.
            struct Index {
                SmallVec<std::pair<const Node*, int>, 64> at;
                int find(const Node* n) const {
                    for (size_t i = 0; i < at.size(); ++i)
                        if (at[i].first == n) return at[i].second;
                    return -1;
                }
                void add(const Node* n, int id) { at.push_back({n, id}); }
                void clear() {
                    while (!at.empty()) at.pop_back();
                }
            };
            Index index_[2];
            bool plan_only_, over_ = false, touched_ = false;
            int visits_ = 0;  // nodes the current add() has walked

            void reindex() {
                index_[0].clear();
                index_[1].clear();
                for (size_t i = 0; i < items.size(); ++i) index_[ctx(items[i])].add(items[i].n.get(), (int)i);
            }
            static int ctx(const Item& x) { return x.leaf ? (x.kept_ctx ? 1 : 0) : x.form == Kept ? 1 : 0; }
            // The form of a shape read right-aligned to S (or, in_kept, to the
            // kept shape).
            Form form_of(const std::vector<int>& s, bool in_kept) const {
                if (!in_kept && s == sp.s) return Full;
                if (!in_kept && s == keep_) return Keep;
                if (in_kept && s == kept_) return Kept;
                for (int d : s)
                    if (d != 1) return None;
                return Scalar;
            }
            Form form_any(const std::vector<int>& s) const {
                const Form f = form_of(s, false);
                return f == None || f == Scalar ? (s == kept_ ? Kept : f) : f;
            }
            bool is_row_reduction(const Node& n) const {
                return ops::is_reduction(n.op) && n.parents[0]->view.shape == sp.s && trailing_axes(n) == sp.k &&
                       (n.view.shape == keep_ || n.view.shape == kept_);
            }
            bool is_column(const Node& n) const {
                return trailing_axes(n, true) == (int)sp.s.size() - sp.k && n.dtype == DType::Float32;
            }
            int held() const {
                int h = 0;
                for (const auto& x : items) h += x.leaf && x.form == Full;
                return h;
            }

            int push(Item x) {
                if ((int)items.size() >= kMaxItems) {
                    over_ = true;
                    return -1;
                }
                items.push_back(std::move(x));
                const int id = (int)items.size() - 1;
                index_[ctx(items[id])].add(items[id].n.get(), id);
                return id;
            }
            // A leaf varies along the row unless it broadcasts over the last k dims.
            int leaf(const NodePtr& n, bool in_kept) {
                Item x;
                x.n = n;
                x.leaf = true;
                x.kept_ctx = in_kept;
                const auto& s = n->view.shape;
                x.form = Scalar;
                for (size_t i = 0; i < s.size(); ++i) {
                    if (s[i] == 1) continue;
                    const bool in_row = !in_kept && s.size() - i <= (size_t)sp.k;
                    x.form = in_row ? Full : x.form == Full ? Full : Keep;
                }
                if (!n->is_realized()) frontier.push_back(n);
                return push(std::move(x));
            }
            int reduce(const NodePtr& n, Form f) {
                if (++reductions > kMaxReductions) {
                    over_ = true;
                    return -1;
                }
                Item x;
                x.n = n;
                x.form = f;
                x.a = visit(n->parents[0], Full);
                return x.a < 0 ? -1 : push(std::move(x));
            }
            // The item of node n read in form `f` (Keep and Full share a context;
            // a node may also turn out to be Scalar). -1 past the limits and for
            // an ARGMAX of the program.
            int visit(const NodePtr& n, Form f) {
                const bool in_kept = f == Kept;
                if (const int id = index_[in_kept].find(n.get()); id >= 0) {
                    // An ARGMAX that is a root here is an integer in the kernel.
                    if (!items[id].leaf && items[id].n->op == OpEnum::ARGMAX) over_ = true;
                    if (over_) return -1;
                    if (items[id].form != Scalar) touched_ = true;
                    return id;
                }
                if (over_) return -1;
                if (++visits_ > kMaxVisits) {
                    over_ = true;
                    return -1;
                }
                if (n->is_realized()) return leaf(n, in_kept);
                Form own = form_of(n->view.shape, in_kept);
                if (f == Keep && own == Full) own = None;
                if (f == Scalar && own != Scalar) own = None;
                if (own == None || (n->device.type != DeviceEnum::HIP && !plan_only_)) return leaf(n, in_kept);
                if (fusible_interior(*n)) {
                    Item x;
                    x.n = n;
                    x.form = own;
                    // A scalar's operands are scalars in either context.
                    const Form cf = own == Scalar && in_kept ? Kept : own;
                    x.a = visit(n->parents[0], cf);
                    if (x.a >= 0 && ops::op_arity(n->op) == 2) x.b = visit(n->parents[1], cf);
                    if (x.a < 0 || (ops::op_arity(n->op) == 2 && x.b < 0)) return -1;
                    if (own == Full)
                        for (int p : {x.a, x.b})
                            if (p >= 0 && !items[p].leaf && (items[p].form == Keep || items[p].form == Kept)) items[p].boundary = true;
                    if (own == Scalar && in_kept) return push_scalar(std::move(x));
                    return push(std::move(x));
                }
                if (n->op == OpEnum::EXPAND) {
                    const NodePtr& p = n->parents[0];
                    if (p->is_realized()) return alias(n, in_kept, leaf_once(p, in_kept));
                    const Form pf = form_of(p->view.shape, in_kept);
                    if (pf == Keep || pf == Scalar) return alias(n, in_kept, visit(p, in_kept ? Kept : Keep));
                    return leaf(n, in_kept);
                }
                if (n->op == OpEnum::RESHAPE) {
                    const NodePtr& p = n->parents[0];
                    if (own == Scalar) return alias(n, in_kept, visit(p, in_kept ? Kept : Keep));
                    if (!p->is_realized() && own == Keep && p->view.shape == kept_) return alias(n, in_kept, visit(p, Kept));
                    if (!p->is_realized() && own == Kept && p->view.shape == keep_) return alias(n, in_kept, visit(p, Keep));
                    return leaf(n, in_kept);
                }
                if ((n->op == OpEnum::SUM || n->op == OpEnum::MAX) && own != Full && own != Scalar && is_row_reduction(*n) &&
                    n->dtype == DType::Float32)
                    return reduce(n, own);
                return leaf(n, in_kept);
            }
            int leaf_once(const NodePtr& p, bool in_kept) {
                if (const int id = index_[in_kept].find(p.get()); id >= 0) {
                    if (items[id].form != Scalar) touched_ = true;
                    return id;
                }
                return leaf(p, in_kept);
            }
            int push_scalar(Item x) {
                const int id = push(std::move(x));
                if (id >= 0) index_[1].add(items[id].n.get(), id);
                return id;
            }
            // Node n (a view) is the value `id` renamed.
            int alias(const NodePtr& n, bool in_kept, int id) {
                if (id >= 0) index_[in_kept].add(n.get(), id);
                return id;
            }
        };

        // The view's source when it only renames a reduction's result.
        const NodePtr& root_of(const NodePtr& r) {
            const NodePtr* n = &r;
            while (!(*n)->is_realized() && (*n)->op == OpEnum::RESHAPE) n = &(*n)->parents[0];
            return *n;
        }

        // The space of a program with this root: a reduction's own, or that of
        // the first row reduction its element-wise region reads.
        bool find_space(const NodePtr& root, Space* sp) {
            if (ops::is_reduction(root->op)) {
                const auto& s = root->parents[0]->view.shape;
                if (const int k = trailing_axes(*root)) return make_space(s, k, sp);
                if (const int j = trailing_axes(*root, true)) return root->op == OpEnum::SUM && make_space(s, (int)s.size() - j, sp);
                return false;
            }
            if (!fusible_interior(*root)) return false;
            bool open = false;
            for (const auto& p : root->parents) open = open || !p->is_realized();
            if (!open) return false;
            SmallSet<Node> seen;
            SmallVec<Node*, 64> stack;
            stack.push_back(root.get());
            int visited = 0;
            while (!stack.empty() && ++visited <= kMaxItems) {
                Node* n = stack.back();
                stack.pop_back();
                for (const auto& p : n->parents) {
                    if (p->is_realized() || !seen.insert(p.get())) continue;
                    if ((p->op == OpEnum::SUM || p->op == OpEnum::MAX)) {
                        const int k = trailing_axes(*p);
                        if (k && make_space(p->parents[0]->view.shape, k, sp)) {
                            const int nd = (int)sp->s.size();
                            const std::vector<int> kept(sp->s.begin(), sp->s.end() - k);
                            std::vector<int> keep = sp->s;
                            for (int d = nd - k; d < nd; ++d) keep[d] = 1;
                            const auto& rs = root->view.shape;
                            if (rs == sp->s || rs == kept || rs == keep) return true;
                        }
                    } else if (fusible_interior(*p) || p->op == OpEnum::EXPAND || p->op == OpEnum::RESHAPE) {
                        stack.push_back(p.get());
                    }
                }
            }
            return false;
        }

        Leaf row_leaf(const Item& x, const Space& sp, bool plan_only) {
            if (!x.kept_ctx) return make_leaf(x.n, sp.s, plan_only);
            Leaf L = make_leaf(x.n, std::vector<int>(sp.s.begin(), sp.s.end() - sp.k), plan_only);
            L.st.resize(sp.s.size(), 0);
            return L;
        }

        // The kernel IR of a program whose leaves are realized, and the nodes
        // its outputs are for (the caller allocates them).
        RowProgram lower(const Builder& b, std::vector<NodePtr>* outs, bool plan_only) {
            RowProgram p;
            p.shape = b.sp.s;
            p.reduced = b.sp.k;
            std::vector<int> value(b.items.size(), -1);
            std::vector<int> insts;
            for (size_t i = 0; i < b.items.size(); ++i) {
                if (!b.items[i].leaf) {
                    insts.push_back((int)i);
                    continue;
                }
                value[i] = (int)p.expr.leaves.size();
                p.expr.leaves.push_back(row_leaf(b.items[i], b.sp, plan_only));
            }
            for (int i : insts) {
                const Item& x = b.items[i];
                Inst in;
                in.op = x.n->op;
                in.a = value[x.a];
                if (x.b >= 0) in.b = value[x.b];
                if (in.op == OpEnum::CAST) in.cast = std::get<CastAttrs>(x.n->attrs).dtype;
                else if (!ops::is_reduction(in.op)) in.lower = HIPLoweringRegistry::find(in.op);
                value[i] = (int)(p.expr.leaves.size() + p.expr.insts.size());
                p.expr.insts.push_back(in);
            }
            SmallSet<Node> stored;
            auto store = [&](const NodePtr& n, int item, RowOut kind) {
                if (!stored.insert(n.get())) return;
                outs->push_back(n);
                p.expr.roots.push_back(value[item]);
                p.out_dtypes.push_back(n->op == OpEnum::ARGMAX ? DType::Int64 : n->dtype);
                p.out_kinds.push_back(kind);
            };
            for (const auto& r : b.roots) {
                const Form f = b.items[r.item].form;
                store(r.n, r.item, r.column ? RowOut::Column : f == Full ? RowOut::Full : RowOut::Row);
            }
            for (int i : insts) {
                const Item& x = b.items[i];
                if (ops::is_reduction(x.n->op) || x.boundary) store(x.n, i, RowOut::Row);
            }
            p.expr.root = p.expr.roots[0];
            return p;
        }

        // Plans and launches a program whose leaves are realized; false (and
        // nothing launched) when the generator declines it.
        bool run(const Builder& b) {
            std::vector<NodePtr> nodes;
            RowProgram p = lower(b, &nodes, false);
            std::vector<std::shared_ptr<Buffer>> bufs;
            for (size_t i = 0; i < nodes.size(); ++i) {
                bufs.push_back(empty(nodes[i]->view.shape, DeviceEnum::HIP, p.out_dtypes[i]));
                p.outs.push_back(bufs.back()->ptr);
            }
            RowPlan plan;
            if (!plan_rows(p, device_compute_units(), &plan, true)) return false;
            std::shared_ptr<Buffer> ws;
            if (plan.two_pass) {
                ws = empty({(int)((plan.workspace_bytes + 3) / 4)}, DeviceEnum::HIP, DType::Float32);
                bind_rows_workspace(plan, ws->ptr);
            }
            launch(plan.first);
            if (plan.two_pass) launch(plan.second);
            // ws returns to the pool here; later work on the stream is ordered
            // after these kernels.
            for (size_t i = 0; i < nodes.size(); ++i) {
                nodes[i]->data = bufs[i];
                nodes[i]->view.strides = calc_contiguous_strides(nodes[i]->view.shape);
            }
            return true;
        }

        // Realizes the leaves of a program over `roots` (of space sp), then the
        // program; false when it is not worthwhile (any more) or declined.
        bool realize_rows(const std::vector<NodePtr>& roots, const Space& sp) {
            for (int attempt = 0; attempt < 4; ++attempt) {
                Builder b(sp);
                for (const auto& r : roots)
                    if (!r->is_realized()) b.add(r);
                if (!b.worthwhile()) return false;
                if (b.frontier.empty()) return run(b);
                for (const auto& f : b.frontier) realize(f);
            }
            return false;
        }
    }  // namespace

    bool row_program_frontier(const NodePtr& root, std::vector<NodePtr>* frontier) {
        Space sp;
        if (!find_space(root, &sp)) return false;
        Builder b(sp);
        if (!b.add(root) || !b.worthwhile()) return false;
        *frontier = std::move(b.frontier);
        return true;
    }

    bool plan_row_program(const std::vector<NodePtr>& roots, int compute_units, RowPlan* plan) {
        Space sp;
        if (roots.empty() || !find_space(roots[0], &sp)) return false;
        Builder b(sp, true);
        for (const auto& r : roots)
            if (!b.add(r)) return false;
        if (!b.worthwhile() || !b.frontier.empty()) return false;
        std::vector<NodePtr> nodes;
        RowProgram p = lower(b, &nodes, true);
        p.outs.assign(nodes.size(), (void*)(uintptr_t)0x100000);
        return plan_rows(p, compute_units, plan);
    }

    bool run_row_program(const NodePtr& root) {
        Space sp;
        return find_space(root, &sp) && realize_rows({root}, sp) && root->is_realized();
    }

    bool starts_row_program(const NodePtr& root) {
        Space sp;
        const NodePtr& n = root_of(root);
        return !n->is_realized() && find_space(n, &sp);
    }

    bool realize_row_groups(const std::vector<NodePtr>& roots) {
        Space sp;
        std::vector<NodePtr> rest;
        SmallSet<Node> seen;
        for (const auto& r : roots) {
            const NodePtr& n = root_of(r);
            if (!n->is_realized() && n->device.type == DeviceEnum::HIP && seen.insert(n.get())) rest.push_back(n);
        }
        bool done = false;
        while (rest.size() >= 2) {
            // The first root that has a space takes every other root that
            // shares operands with it; roots left over start again.
            size_t seed = 0;
            while (seed < rest.size() && !find_space(rest[seed], &sp)) ++seed;
            if (seed == rest.size()) break;
            Builder b(sp);
            std::vector<NodePtr> mine, others(rest.begin(), rest.begin() + seed);
            std::vector<NodePtr> after(rest.begin() + seed + 1, rest.end());
            if (b.add(rest[seed])) mine.push_back(rest[seed]);
            for (auto* list : {&others, &after}) {
                std::vector<NodePtr> left;
                for (const auto& r : *list)
                    if (!mine.empty() && b.add(r)) mine.push_back(r);
                    else left.push_back(r);
                *list = std::move(left);
            }
            if (mine.size() >= 2 && b.worthwhile()) {
                done = true;
                if (b.frontier.empty()) run(b);
                else realize_rows(mine, sp);
            }
            rest = std::move(after);  // what came before the seed has no space of its own
        }
        return done;
    }
}
