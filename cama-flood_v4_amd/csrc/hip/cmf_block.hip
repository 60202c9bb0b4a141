// cmf_block.hip -- many substeps of a model per launch.
//
// The three-phase kernels (cmf_kernels.hip) stream the whole state through HBM on
// every substep and meet the grid between phases. River networks do not need
// that: a cell depends on its neighbours along the river only, two cells
// downstream and two upstream per substep (the limiter rate of a cell needs the
// outflows of its upstream cells, and those their downstream depths). So the
// network is cut into blocks of T cells, one workgroup each, one cell per thread:
// whole basins where they fit, connected parts of larger ones. A block also loads
// the cells within reach of its own over the kmax substeps of a launch and steps
// those redundantly, a shrinking ring of them as the substeps pass, so no block
// waits for another. State lives in registers and LDS between the substeps; HBM
// sees it once per launch. Every value is computed by the statements of the
// three-phase kernels on the same inputs, so results are the same bits.
//
// The levels of a bifurcation path are computed by neighbouring lanes, each keeping
// its flow in a register; the lanes add them up in the order of the levels. That adds
// about a tenth to a substep of a block with 80 paths of 5 levels (as one thread per
// path the five powers and divides in a row would be the longest chain of it).
#include "cmf_block.hpp"

#include <algorithm>
#include <atomic>
#include <new>
#include <queue>
#include <thread>

namespace cmf {

// Whether every basin (total at its mouth), with the basins that paths join to it, is of
// at most T cells: what a closed plan needs.
static bool groups_fit(const BlockNet& net, const std::vector<int32_t>& total, int T) {
    std::vector<int32_t> to((size_t)net.n), size(total);              // a mouth: the mouth it is joined to, or itself
    for (int p = net.n - 1; p >= 0; --p) to[(size_t)p] = net.next[p] >= 0 ? to[(size_t)net.next[p]] : p;
    auto mouth = [&](int p) {
        p = to[(size_t)p];
        while (to[(size_t)p] != p) p = to[(size_t)p] = to[(size_t)to[(size_t)p]];
        return p;
    };
    for (int q = 0; q < net.npth; ++q) {
        if (net.pth_up[q] < 0 || net.pth_down[q] < 0) continue;
        const int a = mouth(net.pth_up[q]), b = mouth(net.pth_down[q]);
        if (a == b) continue;
        to[(size_t)b] = a;
        size[(size_t)a] += size[(size_t)b];
    }
    for (int p = 0; p < net.n; ++p)
        if (to[(size_t)p] == p && size[(size_t)p] > T) return false;
    return true;
}

// What the surroundings ask of a cell, in one place: downstream cell, upstream list, and
// the other ends of its paths (those out of it, then those into it)
struct Node {
    int32_t next, up, end;
    uint16_t nend;
    uint8_t nup;
    bool damup;
};
struct PathEnd { int32_t cell, path; };

// f(0) .. f(nw - 1), on threads of their own where there are any
constexpr int PLAN_THREADS = 4;
template <class F>
static void in_threads(int nw, F f) {
    std::atomic<bool> nomem{false};
    std::atomic<int> next{0};
    auto run = [&] {
        try {
            for (int w = next++; w < nw; w = next++) f(w);
        } catch (const std::bad_alloc&) {
            nomem = true;
        }
    };
    std::vector<std::thread> th;
    try {
        for (int w = 1; w < nw; ++w) th.emplace_back(run);
    } catch (const std::exception&) {
        // no more threads: those there are do it all
    }
    run();
    for (std::thread& t : th) t.join();
    if (nomem) throw std::bad_alloc();
}

// ---------------------------------------------------------------------------
// Partition. Cells come in depth-first order (every cell after its upstream
// subtree). Basins of at most T cells stay whole; larger ones are cut bottom-up
// into connected pieces of at most `cap` cells, so a piece has one downstream cut
// and about one upstream cut. The dependency sets of a piece, r counting the
// substeps that follow in the launch:
//   U_0     = the owned cells
//   R_r     = U_r + upstream(U_r) + downstream(U_r)      limiter rates needed
//   Q_r     = R_r + upstream(R_r)                        outflows needed
//   U_(r+1) = Q_r + downstream(Q_r) + upstream(dam cells of Q_r)
// (a dam's inflow is the previous flow of its upstream cells). code = position of
// the first set a cell is in: U_r <= 3r, R_r <= 3r+1, Q_r <= 3r+2.
//
// Bifurcation paths join cells of different basins: R_r also holds the other ends of
// the paths of U_r (a path is limited at either end), U_(r+1) those of the paths of R_r,
// whose flows R_r needs. The rivers are then cut into small pieces, and a block is
// grown from them along the links, so that most paths stay inside: of 240,019 cells with
// 20,000 paths, 702 blocks of 512 load 1.42 times as many for kmax = 3 and compute 1.22
// times as many outflows (pieces of T/32 cells 780 and 1.58; T/4 710 with more room
// left; without the small pieces put into the room at the end 714).
bool build_block_plan(const BlockNet& net, int T, int kmax, bool closed_only, int64_t max_blocks, BlockPlan& out) {
    const int n = net.n;
    const int32_t *next = net.next, *up_ptr = net.up_ptr, *up_idx = net.up_idx, *domain = net.domain;
    const uint8_t* special = net.special;
    const bool paths = net.npth > 0;
    out = BlockPlan();
    if (n <= 0 || T > (paths ? 512 : 1024) || kmax < 1 || 3 * kmax > (paths ? 60 : 200)) return false;
    if (paths && (net.npthlev < 1 || net.npthlev > 64)) return false;
    const int per_wave = paths ? 64 / net.npthlev : 0;             // paths of a wavefront
    const int max_paths = paths ? std::min(blk_paths(T), per_wave * (T / 64)) : 0;
    const int cap = paths ? std::max(8, T / 8) : std::max(T / 4, T - 48 * kmax);
    std::vector<int32_t> total((size_t)n, 1), resid((size_t)n), piece((size_t)n);
    std::vector<uint8_t> root((size_t)n, 0);
    std::vector<Node> node((size_t)n);
    std::vector<PathEnd> ends;
    if (paths) ends.reserve((size_t)net.out_ptr[n] + (size_t)net.in_ptr[n]);
    for (int p = 0; p < n; ++p) {
        Node& x = node[(size_t)p];
        x = Node{next[p], up_ptr[p], (int32_t)ends.size(), 0, 0, special && (special[p] & BLK_DAMUP)};
        if (paths) {
            const int no = net.out_ptr[p + 1] - net.out_ptr[p], ni = net.in_ptr[p + 1] - net.in_ptr[p];
            if (no > 255 || ni > 255) return false;
            for (int k = net.out_ptr[p]; k < net.out_ptr[p + 1]; ++k) ends.push_back({net.pth_down[net.out_idx[k]], net.out_idx[k]});
            for (int k = net.in_ptr[p]; k < net.in_ptr[p + 1]; ++k) ends.push_back({net.pth_up[net.in_idx[k]], net.in_idx[k]});
            x.nend = (uint16_t)(no + ni);
        }
        if (up_ptr[p + 1] - up_ptr[p] > 250) return false;
        x.nup = (uint8_t)(up_ptr[p + 1] - up_ptr[p]);
        if (next[p] >= 0) {
            if (next[p] <= p) return false;                        // needs the depth-first order
            total[(size_t)next[p]] += total[(size_t)p];
        }
    }
    // basin sizes, then the cuts
    for (int p = n - 1; p >= 0; --p) piece[(size_t)p] = next[p] >= 0 ? piece[(size_t)next[p]] : total[(size_t)p];
    if (closed_only && !groups_fit(net, total, T)) return false;
    bool closed = true;
    for (int p = 0; p < n; ++p) {
        const int lim = !paths && piece[(size_t)p] <= T ? T : cap;
        closed = closed && lim == T;
        int r = 1;
        for (int k = up_ptr[p]; k < up_ptr[p + 1]; ++k)
            if (!root[(size_t)up_idx[k]]) r += resid[(size_t)up_idx[k]];
        while (r > lim) {
            int b = -1;
            for (int k = up_ptr[p]; k < up_ptr[p + 1]; ++k) {
                const int u = up_idx[k];
                if (!root[(size_t)u] && (b < 0 || resid[(size_t)u] > resid[(size_t)b])) b = u;
            }
            root[(size_t)b] = 1;
            r -= resid[(size_t)b];
        }
        resid[(size_t)p] = r;
        if (next[p] < 0) root[(size_t)p] = 1;
    }
    int npc = 0;
    for (int p = n - 1; p >= 0; --p) piece[(size_t)p] = root[(size_t)p] ? npc++ : piece[(size_t)next[p]];
    // owned cells of every piece, ascending
    std::vector<int32_t> off((size_t)npc + 1, 0), own((size_t)n);
    for (int p = 0; p < n; ++p) off[(size_t)piece[(size_t)p] + 1] += 1;
    for (int i = 0; i < npc; ++i) off[(size_t)i + 1] += off[(size_t)i];
    {
        std::vector<int32_t> fill(off.begin(), off.end() - 1);
        for (int p = 0; p < n; ++p) own[(size_t)fill[(size_t)piece[(size_t)p]]++] = p;
    }
    // local cells (owned first) and codes of every piece; a piece whose
    // surroundings overfill a block is halved
    struct Piece { int32_t beg, size, spec, dams, kines, dom, paths; };   // into loc / codes; special cells, paths
    std::vector<Piece> done;
    std::vector<int32_t> loc, mark((size_t)n, -1), cur;
    std::vector<uint8_t> codes, curc;
    loc.reserve((size_t)n + (size_t)n / 4);
    codes.reserve((size_t)n + (size_t)n / 4);
    const int max_spec = blk_special(T);
    const int max_dams = blk_dams(T), max_kines = blk_kines(T);
    auto piece_of = [&](const std::vector<int32_t>& c, size_t from, int count) {
        Piece p{(int32_t)loc.size(), count, 0, 0, 0, domain ? domain[c[from]] : 0, 0};
        for (int j = 0; special && j < count; ++j) {
            const uint8_t f = special[(size_t)c[from + j]];
            p.spec += (f & (BLK_DAM | BLK_LEV)) != 0;
            p.kines += (f & BLK_KINE) != 0;
            p.dams += (f & BLK_DAM) && !(f & BLK_KINE);
        }
        return p;
    };
    auto fits = [&](const Piece& p) {
        return p.size <= T && p.spec <= max_spec && p.dams <= max_dams && p.kines <= max_kines && p.paths <= max_paths;
    };
    int stamp = 0;
    // f(the other end, path) of every path of cell x
    auto each_path = [&](int x, auto f) {
        const Node& c = node[(size_t)x];
        for (int k = c.end; k < c.end + c.nend; ++k) f(ends[(size_t)k].cell, ends[(size_t)k].path);
    };
    // more cells than max_blocks hold
    auto too_many = [&] { return (int64_t)loc.size() > max_blocks * (int64_t)T; };
    // the surroundings of the owned cells in cur, with their codes
    auto surround = [&] {
        const int id = stamp++;
        curc.assign(cur.size(), 0);
        for (int x : cur) mark[(size_t)x] = id;
        auto add = [&](int x) {
            if (x >= 0 && mark[(size_t)x] != id) { mark[(size_t)x] = id; cur.push_back(x); }
        };
        auto add_up = [&](const Node& x) { for (int k = x.up; k < x.up + x.nup; ++k) add(up_idx[k]); };
        auto add_ends = [&](const Node& x) { for (int k = x.end; k < x.end + x.nend; ++k) add(ends[(size_t)k].cell); };
        size_t eu = 0;                                              // members whose neighbours are all in
        for (int r = 0; r < kmax && (int)cur.size() <= T; ++r) {
            const size_t r0 = eu;
            eu = cur.size();
            for (size_t j = r0; j < eu; ++j) {
                const Node& x = node[(size_t)cur[j]];
                add_up(x); add(x.next); add_ends(x);
            }
            const size_t er = cur.size();
            curc.resize(er, (uint8_t)(3 * r + 1));
            for (size_t j = eu; j < er; ++j) add_up(node[(size_t)cur[j]]);
            const size_t eq = cur.size();
            curc.resize(eq, (uint8_t)(3 * r + 2));
            for (size_t j = eu; j < eq; ++j) {
                const Node& x = node[(size_t)cur[j]];
                add(x.next);
                if (x.damup) add_up(x);
            }
            for (size_t j = eu; paths && j < er; ++j) add_ends(node[(size_t)cur[j]]);
            curc.resize(cur.size(), (uint8_t)(3 * r + 3));
            eu = er;
        }
    };
    // paths whose flows a cell of this code asks for, from its set R_r on (kmax: none)
    auto path_step = [&](int code) { return std::min(kmax, code < 2 ? 0 : (code + 1) / 3); };
    std::vector<int32_t> pmark(paths ? (size_t)net.npth : 0, -1);
    auto count_paths = [&] {
        const int id = stamp++;
        int m = 0;
        for (size_t j = 0; j < cur.size(); ++j)
            if (path_step(curc[j]) < kmax)
                each_path(cur[j], [&](int, int q) { if (pmark[(size_t)q] != id) { pmark[(size_t)q] = id; ++m; } });
        return m;
    };
    auto keep = [&](Piece pc, int nown) {
        done.push_back(pc);
        closed = closed && (int)cur.size() == nown;
        loc.insert(loc.end(), cur.begin(), cur.end());
        codes.insert(codes.end(), curc.begin(), curc.end());
    };
    if (paths) {
        closed = true;
        // blocks grown from the river pieces: always the one with most links to the
        // block for its size, from a seed with most links to the blocks before
        std::vector<int32_t> links((size_t)npc, 0), seen((size_t)npc, -1), before((size_t)npc, 0), took, grown;
        std::vector<uint8_t> in((size_t)npc, 0);
        typedef std::pair<float, int32_t> Cand;
        std::priority_queue<Cand> near, seeds;
        int first = 0, blk = 0;
        double share = 0.8;                                         // owned cells of a full block
        auto size_of = [&](int i) { return off[(size_t)i + 1] - off[(size_t)i]; };
        auto each_link = [&](int i, auto f) {                       // pieces a piece is joined to
            for (int e = off[(size_t)i]; e < off[(size_t)i + 1]; ++e) {
                const int x = own[(size_t)e];
                auto to = [&](int y) { if (y >= 0 && piece[(size_t)y] != i && !in[(size_t)piece[(size_t)y]]) f(piece[(size_t)y]); };
                const Node& c = node[(size_t)x];
                to(c.next);
                for (int k = c.up; k < c.up + c.nup; ++k) to(up_idx[k]);
                each_path(x, [&](int y, int) { to(y); });
            }
        };
        auto take = [&](int i) {
            in[(size_t)i] = 1;
            took.push_back(i);
            each_link(i, [&](int c) {
                if (seen[(size_t)c] != blk) { seen[(size_t)c] = blk; links[(size_t)c] = 0; }
                links[(size_t)c] += 1;
                near.push({(float)links[(size_t)c] / (float)size_of(c), c});
            });
        };
        std::vector<int32_t> best;
        std::vector<uint8_t> best_codes;
        for (int left = npc; left > 0; ++blk) {
            took.clear();
            grown.clear();
            while (!near.empty()) near.pop();
            int target = std::max(1, (int)(share * T));
            bool shrunk = false;
            for (int tries = 0;; ++tries) {
                while (!shrunk && (int)grown.size() < target && left > (int)took.size()) {
                    int i = -1;
                    while (!near.empty() && i < 0) {
                        const int c = near.top().second;
                        near.pop();
                        if (!in[(size_t)c]) i = c;
                    }
                    while (i < 0 && took.empty() && !seeds.empty()) {
                        if (!in[(size_t)seeds.top().second]) i = seeds.top().second;
                        seeds.pop();
                    }
                    for (int f = first; i < 0; ++f)
                        if (!in[(size_t)f]) i = f;
                        else if (f == first) ++first;
                    if (!grown.empty() && (int)grown.size() + size_of(i) > T) break;
                    grown.insert(grown.end(), own.begin() + off[(size_t)i], own.begin() + off[(size_t)i + 1]);
                    take(i);
                }
                cur = grown;
                surround();
                Piece pc = piece_of(cur, 0, (int)cur.size());
                pc.paths = count_paths();
                const bool ok = fits(pc);
                const bool full = left == (int)took.size() || cur.size() > 0.96 * T || tries >= 4 || shrunk ||
                                  pc.spec > 0.9 * max_spec || pc.dams > 0.9 * max_dams || pc.paths > 0.94 * max_paths;
                if (ok && full) {
                    // small pieces into the room that is left
                    for (int more = 0; more < 6 && !near.empty(); ++more) {
                        const int room = T - pc.size;
                        int i = -1;
                        while (!near.empty() && i < 0 && room > T / 64) {
                            const int c = near.top().second;
                            near.pop();
                            if (!in[(size_t)c] && 4 * size_of(c) <= 3 * room) i = c;
                        }
                        if (i < 0) break;
                        best.swap(cur);
                        best_codes.swap(curc);
                        const size_t had = grown.size();
                        grown.insert(grown.end(), own.begin() + off[(size_t)i], own.begin() + off[(size_t)i + 1]);
                        cur = grown;
                        surround();
                        Piece with = piece_of(cur, 0, (int)cur.size());
                        with.paths = count_paths();
                        if (fits(with)) {
                            pc = with;
                            take(i);
                        } else {
                            grown.resize(had);
                            cur.swap(best);
                            curc.swap(best_codes);
                        }
                    }
                    share = std::max(0.1, std::min(1.0, (double)grown.size() / T));
                    keep(pc, (int)grown.size());
                    if (too_many()) return false;
                    break;
                }
                if (ok) {                                           // room for more
                    target = std::max((int)grown.size() + 1, (int)((double)grown.size() * 0.985 * T / (double)cur.size()));
                    continue;
                }
                // too much: the pieces taken last go back, one at least
                if (took.size() < 2) return false;
                target = (int)std::min((double)grown.size() * 0.96, (double)grown.size() * 0.97 * T / (double)cur.size());
                while (took.size() > 1 && (int)grown.size() > target) {
                    const int i = took.back();
                    took.pop_back();
                    grown.resize(grown.size() - (size_t)size_of(i));
                    in[(size_t)i] = 0;
                    first = std::min(first, i);
                }
                shrunk = true;
            }
            left -= (int)took.size();
            for (int i : took)
                each_link(i, [&](int c) {
                    before[(size_t)c] += 1;
                    seeds.push({(float)before[(size_t)c] / (float)size_of(c), c});
                });
        }
    }
    std::vector<std::vector<int32_t>> work;
    if (paths) npc = 0;                                             // all of them are in blocks
    for (int i = 0; i < npc; ++i) {
        const int a = off[(size_t)i], b = off[(size_t)i + 1], rt = own[(size_t)b - 1];
        const Piece whole = piece_of(own, (size_t)a, b - a);
        if (next[rt] < 0 && total[(size_t)rt] == b - a && fits(whole)) {   // a whole basin
            done.push_back(whole);
            loc.insert(loc.end(), own.begin() + a, own.begin() + b);
            codes.insert(codes.end(), (size_t)(b - a), (uint8_t)0);
            continue;
        }
        work.assign(1, std::vector<int32_t>(own.begin() + a, own.begin() + b));
        while (!work.empty()) {
            cur.swap(work.back());
            work.pop_back();
            const int nown = (int)cur.size();
            surround();
            const Piece pc = piece_of(cur, 0, (int)cur.size());
            if (fits(pc)) {
                keep(pc, nown);
                if (too_many()) return false;
                continue;
            }
            if (nown < 2) return false;
            // halve: cut above the cell whose subtree inside the piece is nearest to half
            cur.resize((size_t)nown);
            const int idp = stamp++;
            for (int x : cur) { mark[(size_t)x] = idp; resid[(size_t)x] = 1; }
            int best = -1, bd = n;
            for (int x : cur) {
                const int d = std::abs(2 * resid[(size_t)x] - nown);
                if (x != cur.back() && d < bd) { bd = d; best = x; }
                if (next[x] >= 0 && mark[(size_t)next[x]] == idp) resid[(size_t)next[x]] += resid[(size_t)x];
            }
            std::vector<int32_t> lo, hi;
            const int idh = stamp++;
            for (int j = nown - 1; j >= 0; --j) {
                const int x = cur[(size_t)j];
                if (x == best || (next[x] >= 0 && mark[(size_t)next[x]] == idh)) mark[(size_t)x] = idh;
            }
            for (int x : cur) (mark[(size_t)x] == idh ? hi : lo).push_back(x);
            work.push_back(std::move(lo));
            work.push_back(std::move(hi));
        }
    }
    // pieces into blocks: the large ones best-fit by descending size, the small
    // ones fill the room that is left, in order
    std::vector<std::vector<int32_t>> bins;
    std::vector<Piece> room;                                       // what is left in each
    {
        auto holds = [](const Piece& r, const Piece& p) {
            return r.dom == p.dom && r.size >= p.size && r.spec >= p.spec && r.dams >= p.dams && r.kines >= p.kines &&
                   r.paths >= p.paths;
        };
        auto put = [&](int b, size_t k) {
            if (b < 0) {
                b = (int)bins.size();
                bins.emplace_back();
                room.push_back({0, T, max_spec, max_dams, max_kines, done[k].dom, max_paths});
                out.dom.push_back(done[k].dom);
            }
            const Piece& p = done[k];
            Piece& r = room[(size_t)b];
            bins[(size_t)b].push_back((int32_t)k);
            r.size -= p.size; r.spec -= p.spec; r.dams -= p.dams; r.kines -= p.kines; r.paths -= p.paths;
            return b;
        };
        // domain by domain (the pieces were cut in descending cell order)
        std::vector<int32_t> ord(done.size());
        for (size_t k = 0; k < ord.size(); ++k) ord[k] = (int32_t)k;
        std::stable_sort(ord.begin(), ord.end(), [&](int32_t x, int32_t y) { return done[(size_t)x].dom < done[(size_t)y].dom; });
        std::vector<std::vector<int32_t>> by_size((size_t)T + 1), by_room((size_t)T + 1);
        const int small = T / 16;
        for (size_t o0 = 0, o1 = 0; o0 < ord.size(); o0 = o1) {
            while (o1 < ord.size() && done[(size_t)ord[o1]].dom == done[(size_t)ord[o0]].dom) ++o1;
            for (auto& v : by_size) v.clear();
            for (auto& v : by_room) v.clear();
            const size_t first = bins.size();
            for (size_t o = o0; o < o1; ++o)
                if (done[(size_t)ord[o]].size > small) by_size[(size_t)done[(size_t)ord[o]].size].push_back(ord[o]);
            for (int s = T; s > small; --s)
                for (int32_t k : by_size[(size_t)s]) {
                    int b = -1;
                    for (int r = s; r <= T && b < 0; ++r)
                        if (!by_room[(size_t)r].empty() && holds(room[(size_t)by_room[(size_t)r].back()], done[(size_t)k])) {
                            b = by_room[(size_t)r].back();
                            by_room[(size_t)r].pop_back();
                        }
                    b = put(b, (size_t)k);
                    by_room[(size_t)room[(size_t)b].size].push_back(b);
                }
            size_t b = first;
            for (size_t o = o0; o < o1; ++o) {
                const size_t k = (size_t)ord[o];
                if (done[k].size > small) continue;
                while (b < bins.size() && !holds(room[b], done[k])) ++b;
                put(b < bins.size() ? (int)b : -1, k);
            }
        }
    }
    // in the order of their cells, as neighbours share lines of the state
    std::sort(bins.begin(), bins.end(), [&](const std::vector<int32_t>& x, const std::vector<int32_t>& y) {
        return loc[(size_t)done[(size_t)x[0]].beg] < loc[(size_t)done[(size_t)y[0]].beg];
    });
    for (size_t b = 0; b < bins.size(); ++b) out.dom[b] = done[(size_t)bins[b][0]].dom;
    const int nb = (int)bins.size();
    if ((closed_only && !closed) || nb > max_blocks) return false;
    const size_t np = (size_t)nb * (size_t)T;
    out.T = T; out.kmax = kmax; out.nblk = nb; out.closed = closed;
    out.cell.assign(np, -1);
    out.topo.assign(2 * np, 0);
    out.upx_ptr.assign(np, 0);
    out.ndam.assign((size_t)nb, 0);
    const size_t npb = (size_t)blk_paths(T);
    if (paths) {
        out.path.assign(np, -1);
        out.pword.assign(np, 0);
        out.pcell.assign(np, 0);
        out.ppx_ptr.assign(np, 0);
        out.pends.assign((size_t)nb * npb, 0);
    }
    // Tables of blocks `from` to `to` - 1; the lists of the cells with more than two upstream
    // cells or paths go to upx and ppx. Order inside a block: dam, kinematic and levee cells
    // in places of their own (their wavefronts take the rare paths, the others never do),
    // then the owned cells, then the ring by code.
    auto tables = [&](int from, int to, std::vector<uint16_t>& upx, std::vector<uint16_t>& ppx) {
        std::vector<int32_t> pos((size_t)n), in((size_t)n, -1);        // place in the block, piece it is of
        std::vector<int32_t> slot(pmark.size()), slot_of(pmark.size(), -1);
        std::vector<int32_t> place((size_t)T), count((size_t)3 * kmax + 6), spot((size_t)T);
        std::vector<std::pair<int, int>> plist;                        // code, path
        auto code_of = [&](size_t e) { return closed ? 0 : (int)codes[e]; };
        auto key_of = [&](size_t e) {
            const uint8_t f = special ? special[(size_t)loc[e]] : 0;
            return f & BLK_KINE ? 1 : (f & BLK_DAM ? 0 : (f & BLK_LEV ? 2 : 3 + code_of(e)));
        };
        for (int b = from; b < to; ++b) {
            const std::vector<int32_t>& bin = bins[(size_t)b];
            std::fill(count.begin(), count.end(), 0);
            for (int32_t k : bin)
                for (int j = 0; j < done[(size_t)k].size; ++j) count[(size_t)key_of((size_t)done[(size_t)k].beg + j) + 1] += 1;
            const int na = count[1], nk = count[2];
            out.ndam[(size_t)b] = na | (nk << 16);
            for (size_t i = 0; i + 1 < count.size(); ++i) count[i + 1] += count[i];
            // spot[rank in that order] = place
            for (int i = 0; i < na; ++i) spot[(size_t)i] = i;
            for (int i = 0; i < nk; ++i) spot[(size_t)(na + i)] = BLK_KINE_AT + i;
            for (int i = na + nk, l = na; i < T; ++i, ++l) {
                if (nk > 0 && l == BLK_KINE_AT) l += nk;
                spot[(size_t)i] = l;
            }
            int q = 0;
            for (int32_t k : bin)
                for (int j = 0; j < done[(size_t)k].size; ++j, ++q)
                    place[(size_t)q] = spot[(size_t)count[(size_t)key_of((size_t)done[(size_t)k].beg + j)]++];
            q = 0;
            int slots = 0;
            for (int32_t k : bin) {
                const Piece& pc = done[(size_t)k];
                // a piece's neighbours are looked up inside the piece: two pieces of one
                // block may both hold a cell
                for (int j = 0; j < pc.size; ++j) {
                    const int x = loc[(size_t)pc.beg + j];
                    in[(size_t)x] = k;
                    pos[(size_t)x] = place[(size_t)(q + j)];
                }
                if (paths) {
                    // slots of the paths, the owner's (of the upstream end) first; two
                    // pieces of one block may both have a path
                    plist.clear();
                    for (int j = 0; j < pc.size; ++j) {
                        const int x = loc[(size_t)pc.beg + j], step = path_step(code_of((size_t)pc.beg + j));
                        const bool mine = codes[(size_t)pc.beg + j] == 0;
                        if (step < kmax)
                            each_path(x, [&](int, int w) {
                                const int code = mine && net.pth_up[w] == x ? 0 : 3 * step + 2;
                                if (slot_of[(size_t)w] != k) {
                                    slot_of[(size_t)w] = k;
                                    slot[(size_t)w] = (int)plist.size();
                                    plist.push_back({code, w});
                                } else {
                                    int& c = plist[(size_t)slot[(size_t)w]].first;
                                    c = std::min(c, code);
                                }
                            });
                    }
                    std::stable_sort(plist.begin(), plist.end(),
                                     [](const std::pair<int, int>& x, const std::pair<int, int>& y) { return x.first < y.first; });
                    for (const auto& cw : plist) {
                        const int w = cw.second, sl = slots++;
                        slot[(size_t)w] = sl;
                        out.pends[(size_t)b * npb + sl] = (uint32_t)pos[(size_t)net.pth_up[w]] | ((uint32_t)pos[(size_t)net.pth_down[w]] << 10);
                        for (int v = 0; v < net.npthlev; ++v) {
                            const size_t e = (size_t)b * T + (size_t)(T - 64 * (1 + sl / per_wave) + sl % per_wave * net.npthlev + v);
                            out.path[e] = w;
                            out.pword[e] = (uint32_t)v | ((uint32_t)sl << PATH_SLOT) | ((uint32_t)(closed ? 0 : cw.first) << PATH_CODE);
                        }
                    }
                }
                for (int j = 0; j < pc.size; ++j, ++q) {
                    const int x = loc[(size_t)pc.beg + j];
                    const int code = code_of((size_t)pc.beg + j);
                    const size_t e0 = (size_t)b * T + place[(size_t)q];
                    uint32_t nx = TOPO_MOUTH;
                    if (next[x] >= 0) {
                        const bool inside = in[(size_t)next[x]] == k;
                        if (!inside && code <= 3 * (kmax - 1) + 2) return false;   // cannot be
                        nx = inside ? (uint32_t)pos[(size_t)next[x]] : (uint32_t)place[(size_t)q];
                    }
                    int nup = up_ptr[x + 1] - up_ptr[x];
                    for (int e = up_ptr[x]; e < up_ptr[x + 1]; ++e)
                        if (in[(size_t)up_idx[e]] != k) {
                            if (code <= 3 * (kmax - 1) + 1) return false;          // cannot be
                            nup = 0;                                      // never asked for
                            break;
                        }
                    const uint32_t u0 = nup > 0 ? (uint32_t)pos[(size_t)up_idx[up_ptr[x]]] : 0u;
                    const uint32_t u1 = nup > 1 ? (uint32_t)pos[(size_t)up_idx[up_ptr[x] + 1]] : u0;
                    const uint32_t fl = special ? special[(size_t)x] & (BLK_DAM | BLK_LEV) : 0u;
                    out.cell[e0] = x;
                    out.topo[e0] = nx | (u0 << TOPO_UP0) | (fl << TOPO_FLAGS);
                    out.topo[np + e0] = u1 | ((uint32_t)nup << TOPO_NUP) | ((uint32_t)code << TOPO_CODE);
                    if (paths && path_step(code) < kmax) {
                        const int no = net.out_ptr[x + 1] - net.out_ptr[x], ni = net.in_ptr[x + 1] - net.in_ptr[x];
                        uint32_t w = ((uint32_t)no << 16) | ((uint32_t)ni << 24);
                        int at = 0;
                        if (no + ni > 2) out.ppx_ptr[e0] = (int32_t)ppx.size();
                        each_path(x, [&](int, int p) {
                            if (at < 2) w |= (uint32_t)slot[(size_t)p] << (8 * at);
                            else ppx.push_back((uint16_t)slot[(size_t)p]);
                            ++at;
                        });
                        out.pcell[e0] = w;
                    }
                    if (nup > 2) {
                        out.upx_ptr[e0] = (int32_t)upx.size();
                        for (int e = up_ptr[x] + 2; e < up_ptr[x + 1]; ++e)
                            upx.push_back((uint16_t)pos[(size_t)up_idx[e]]);
                    }
                }
            }
            for (int l = 0; l < T; ++l)
                if (out.cell[(size_t)b * T + l] < 0) out.topo[np + (size_t)b * T + l] = 255u << TOPO_CODE;   // idle
        }
        return true;
    };
    // in a few ranges of blocks, then their lists one after another
    const int nr = nb < 64 ? 1 : PLAN_THREADS;
    std::vector<std::vector<uint16_t>> upx((size_t)nr), ppx((size_t)nr);
    std::atomic<bool> ok{true};
    auto range = [&](int r) { return (int)((int64_t)nb * r / nr); };
    in_threads(nr, [&](int r) {
        if (!tables(range(r), range(r + 1), upx[(size_t)r], ppx[(size_t)r])) ok = false;
    });
    if (!ok) return false;
    out.upx.swap(upx[0]);
    out.ppx.swap(ppx[0]);
    for (int r = 1; r < nr; ++r) {
        const int32_t du = (int32_t)out.upx.size(), dp = (int32_t)out.ppx.size();
        for (size_t e = (size_t)range(r) * (size_t)T; e < (size_t)range(r + 1) * (size_t)T; ++e) {
            if (((out.topo[np + e] >> TOPO_NUP) & 0xff) > 2) out.upx_ptr[e] += du;
            if (paths && ((out.pcell[e] >> 16) & 0xff) + (out.pcell[e] >> 24) > 2) out.ppx_ptr[e] += dp;
        }
        out.upx.insert(out.upx.end(), upx[(size_t)r].begin(), upx[(size_t)r].end());
        out.ppx.insert(out.ppx.end(), ppx[(size_t)r].begin(), ppx[(size_t)r].end());
    }
    if (out.upx.empty()) out.upx.push_back(0);
    if (out.ppx.empty()) out.ppx.push_back(0);
    return true;
}

// ---------------------------------------------------------------------------
// Values of the cells of a block between the phases and substeps. With FP64 state
// the arrays of T cells take 120 bytes a cell and the first NL floodplain heights 20
// more, which fills the 160 KB of a CU with 1024 cells; the mixed form has room for
// all heights. With paths and levees or dams there is room for one, if two blocks of 512
// cells are to share a CU.
template <class R, int T, bool LEV, bool DAM, bool PTH>
struct BlockLds {
    static constexpr bool kOutSum = sizeof(R) == sizeof(float);
    static constexpr int NL = kOutSum ? 8 : (PTH && (LEV || DAM) ? 1 : 5), NS = blk_special(T), ND = blk_dams(T) + blk_kines(T);
    static constexpr int NP = PTH ? blk_paths(T) : 1;
    R dph[T], dphp[T], q[T], f[T], rate[T];    // read by neighbours
    R fpre[T], fdph[T], ffrc[T];               // own floodplain state
    R a_riv[T], a_fld[T], a_vel[T], a_out[kOutSum ? 1 : T], m_out[T], m_dph[T], m_sto[T];
    float hgt[NL][T];
    double sum[2 * NGLB * (T / 64)];
    // dam and kinematic cells (slot_of_dam), levee cells
    double dam[DAM ? ND : 1], daminf[DAM ? ND : 1], vk[DAM ? ND : 1], vf[DAM ? ND : 1];
    R a_inf[DAM ? ND : 1], ro[DAM ? ND : 1], fo[DAM ? ND : 1];   // average of DAMINF; limited flows, read downstream
    int32_t drow[DAM ? ND : 1], dcode[DAM ? ND : 1];
    double lev[LEV ? NS : 1];
    int32_t lrow[LEV ? NS : 1];
    // paths: STORGE of the cells, flow of a path summed over its levels and its ends, LEVDPH
    R sto[PTH ? T : 1], psum[NP], ldph[PTH && LEV ? NS : 1];
    uint32_t pend[NP];
};
enum { DAM_CODE = 15, DAM_KINE = 16, DAM_ACTIVE = 32, DAM_BALANCE = 64 };   // bits of dcode (I1DAM below)
__device__ __forceinline__ int slot_of_dam(int l, int T) { return l < BLK_KINE_AT ? l : l - BLK_KINE_AT + blk_dams(T); }
template <int NL, int T>
struct BlockHgt {
    const float *s, *h;
    int n;
    __device__ __forceinline__ float operator()(int l) const {
        return l <= NL ? s[(l - 1) * T] : h[(size_t)(l - 1) * n];
    }
    __device__ __forceinline__ const BlockHgt& row() const { return *this; }
};

template <class R>
struct BlockArgs {
    DevMap M;
    DevState<R> S;
    BlockState<R> O;
    BlockTab P;
    StepArgs A;
    InstStep I;
    int j;
    const R* vel0;
};

// The kernel's arguments, re-read through an opaque pointer: the substep loop is
// long, and pointers and constants loaded once for all of it would not fit the
// scalar registers (they would spill into vector lanes); a scalar load where one
// is used hits the constant cache.
template <class R>
__device__ __forceinline__ const BlockArgs<R>& block_args() {
    typedef const __attribute__((address_space(4))) BlockArgs<R>* cptr;
    cptr p = (cptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const BlockArgs<R>*)p;
}

// Workgroup barrier for data in LDS only: loads and stores of global memory stay in
// flight across it (a full barrier waits for them, the runoff of the update and the
// budget sums among them).
__device__ __forceinline__ void sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <class R, int T, bool LEV, bool DAM, bool MB, bool PTH>
__global__ __launch_bounds__(T, sizeof(R) == 4 && T < 1024 ? 6 : 4) void k_block(BlockArgs<R> args_) {
    constexpr bool kOutSum = sizeof(R) == sizeof(float);
    constexpr int NW = T / 64;
    // budget terms formed before the stage inversion (STOPRE2 is STONEW in FP64) and after it
    constexpr int NA = kOutSum ? G_STOPRE2 + 1 : G_STOPRE2, NB = (LEV ? NGLB : G_LEVSTO) - G_STONEW2;
    __shared__ BlockLds<R, T, LEV, DAM, PTH> L;
    int l = threadIdx.x, b = blockIdx.x, m = 0;
    int nt = args_.I.nt;
    double dt = args_.I.dt, gdt = args_.I.gdt;
    if (MB) {
        // the members of a block of cells follow each other on one XCD (consecutive
        // workgroups go round the eight), as they share the lines of its state
        const int lgm = args_.M.lgm, r = b >> 3;
        m = r & ((1 << lgm) - 1);
        b = ((r >> lgm) << 3) + (b & 7);
        if (b >= args_.P.nblk) return;
        const InstStep& I = args_.S.inst[(args_.P.dom[b] << lgm) + m];
        nt = I.nt; dt = I.dt; gdt = I.gdt;
    } else {
        // neighbouring blocks on one XCD, as they share lines of the state: 240,019 cells
        // with 20,000 paths 64.2 -> 62.9 ms (not for ensembles, whose instances of few
        // substeps would leave their XCD idle: 38.5 -> 45.9)
        b = (b & 7) * ((args_.P.nblk + 7) >> 3) + (b >> 3);
        if (b >= args_.P.nblk) return;
    }
    const int nl = block_launches(nt, args_.P.kmax, args_.P.closed);
    if (MB && (nt < 1 || args_.j >= nl)) return;                          // done, or no substep to take
    const int it0 = (int)((long long)nt * args_.j / nl), nsub = (int)((long long)nt * (args_.j + 1) / nl) - it0;
    int g, s0;                                                            // cell, state slot
    uint32_t w0, w1;
    const R zero = R(0);
    double rs = 0.0, fs = 0.0, zdn = 0.0;
    R ro = zero, fo = zero;
    int gp = -1;                                                          // path of this thread's level
    uint32_t wp = 0, wc = 0;
    R pf = zero;                                                          // its flow
    float f_elevtn = 0.f, f_nxtdst = 1.f, f_rivman = 1.f, f_rivlen = 1.f, f_rivwth = 1.f, f_grarea = 1.f, f_rivhgt = 1.f;
    {
        const BlockArgs<R>& a = block_args<R>();
        const DevMap& M = a.M;
        const DevState<R>& S = a.S;
        const BlockTab& P = a.P;
        const int pl = b * T + l;
        g = P.cell[pl];
        s0 = MB ? (g << M.lgm) | m : g;
        w0 = P.topo[pl];
        w1 = P.topo[(size_t)P.nblk * T + pl];
        const bool mouth = (w0 & TOPO_MOUTH) == TOPO_MOUTH;
        using Lds = BlockLds<R, T, LEV, DAM, PTH>;
        if (g >= 0) {
            rs = S.rivsto[s0]; fs = S.fldsto[s0];
            ro = S.rivout[s0]; fo = S.fldout[s0];
            L.dph[l] = S.rivdph[s0]; L.dphp[l] = S.rivdph_pre[s0];
            L.fpre[l] = S.fldsto_pre[s0]; L.fdph[l] = S.flddph[s0]; L.ffrc[l] = S.fldfrc[s0];
            f_rivlen = M.rivlen[g]; f_rivwth = M.rivwth[g]; f_grarea = M.grarea[g]; f_rivhgt = M.rivhgt[g];
            f_elevtn = M.elevtn[g]; f_nxtdst = M.nxtdst[g]; f_rivman = M.rivman[g];
            if (mouth) zdn = M.dwnelv[g];
#pragma unroll
            for (int k = 0; k < Lds::NL; ++k)
                if (k < M.nlfp) L.hgt[k][l] = M.fldhgt[(size_t)k * M.n + g];
            if (LEV && (w0 & (BLK_LEV << TOPO_FLAGS))) { L.lev[l] = S.levsto[s0]; L.lrow[l] = M.lev_idx[g]; }
            if (DAM && (w0 & (BLK_DAM << TOPO_FLAGS))) {
                const int e = slot_of_dam(l, T);
                const int c = M.i1dam[g], d = M.dam_of_cell[g];
                int bits = c > 0 ? c & DAM_CODE : 0;
                if (c == 10 && !mouth) {
                    bits |= DAM_KINE;
                    double vk, vf;
                    dam_kine_factors(M, a.A.pminslp, a.A.pmanfld, g, M.next[g], vk, vf);
                    L.vk[e] = vk; L.vf[e] = vf;
                }
                if (d >= 0 && M.damstat[d] > 0) bits |= DAM_ACTIVE;
                if (d >= 0 && M.damstat[d] != -9999) bits |= DAM_BALANCE;
                L.dcode[e] = bits; L.drow[e] = d;
                const bool mine = (w1 >> TOPO_CODE) == 0;
                L.dam[e] = S.damsto[s0]; L.daminf[e] = mine ? S.daminf[s0] : 0.0;
                L.a_inf[e] = mine && it0 > 0 ? S.daminf_avg[s0] : zero;
                L.ro[e] = ro; L.fo[e] = fo;
            }
        }
        if (PTH) {
            if (g >= 0) {
                wc = P.pcell[pl];
                double st = rs + fs;
                if (LEV && (w0 & (BLK_LEV << TOPO_FLAGS))) { st = st + L.lev[l]; L.ldph[l] = S.levdph[s0]; }
                L.sto[l] = R(st);
            }
            gp = P.path[pl];
            if (gp >= 0) {
                wp = P.pword[pl];
                const int lev = (int)(wp & 63u), slot = (int)(wp >> PATH_SLOT) & 0xff;
                pf = S.pthflw[(size_t)lev * M.nsp + gp];
                if (lev == 0) {
                    const int ip = M.pth_upst[gp], jp = M.pth_down[gp], mi = M.i2mask[ip], mj = M.i2mask[jp];
                    uint32_t pe = P.pends[(size_t)b * Lds::NP + slot];
                    if (LEV ? mi == 1 || mj == 1 : mi > 0 || mj > 0) pe |= END_SKIP;
                    if (mi > 0 || mj > 0) pe |= END_NOLIM;                  // inflow_lspamat:501
                    if (LEV) {
                        const int u = M.lev_idx[ip], v = M.lev_idx[jp];
                        if (u >= 0 && M.lev_tab[M.nlevcell + u] < 1.0) pe |= END_LEV_I;
                        if (v >= 0 && M.lev_tab[M.nlevcell + v] < 1.0) pe |= END_LEV_J;
                    }
                    L.pend[slot] = pe;
                }
            }
        }
        const bool cont = (w1 >> TOPO_CODE) == 0 && it0 > 0;
        L.a_riv[l] = cont ? S.rivout_avg[s0] : zero;
        L.a_fld[l] = cont ? S.fldout_avg[s0] : zero;
        L.a_vel[l] = cont ? S.rivvel_avg[s0] : zero;
        if (!kOutSum) L.a_out[l] = cont ? S.outflw_avg[s0] : zero;
        L.m_out[l] = cont ? S.outflw_max[s0] : zero;
        L.m_dph[l] = cont ? S.rivdph_max[s0] : zero;
        L.m_sto[l] = cont ? S.storge_max[s0] : zero;
        // the downstream cell's bed, through LDS
        L.q[l] = R(f_elevtn); L.f[l] = R(f_rivhgt);
        sync_lds();
        if (!mouth) {
            const int nx = (int)(w0 & TOPO_MOUTH);
            zdn = (double)L.q[nx] - (double)L.f[nx];
        }
    }
    sync_lds();
    for (int s = 0; s < nsub; ++s) {
        // what follows from these is formed anew in every substep: kept across the
        // loop it would take twice the registers there are
        asm volatile("" : "+v"(f_elevtn), "+v"(f_nxtdst), "+v"(f_rivman), "+v"(f_rivlen), "+v"(f_rivwth), "+v"(f_grarea),
                     "+v"(f_rivhgt), "+v"(w0), "+v"(w1), "+v"(g), "+v"(l));
        if (MB) asm volatile("" : "+v"(s0));
        if (PTH) asm volatile("" : "+v"(gp), "+v"(wp), "+v"(wc));
        const BlockArgs<R>& a = block_args<R>();
        const DevMap& M = a.M;
        const DevState<R>& S = a.S;
        const BlockTab& P = a.P;
        const StepArgs& A = a.A;
        const R rdt = R(dt);
        const int nx = (int)(w0 & TOPO_MOUTH);
        const bool river = nx != (int)TOPO_MOUTH;
        const int u0 = (int)(w0 >> TOPO_UP0) & 0x3ff, u1 = (int)(w1 & 0x3ffu), nup = (int)(w1 >> TOPO_NUP) & 0xff;
        // an idle lane is in no set, however many substeps remain
        const int code = g < 0 ? 0x7fffffff : (int)(w1 >> TOPO_CODE);
        const bool own = code == 0;
        const bool is_dam = DAM && (w0 & (BLK_DAM << TOPO_FLAGS));
        const int e = slot_of_dam(l, T);
        const bool is_lev = LEV && (w0 & (BLK_LEV << TOPO_FLAGS));
        const int it = it0 + s, rem = nsub - 1 - s;
        const bool last = it == nt - 1;
        // ---- path flows, a level per lane (pthflow_path)
        if (PTH && __any(gp >= 0 && (int)(wp >> PATH_CODE) <= 3 * rem + 2)) {
            const bool act = gp >= 0 && (int)(wp >> PATH_CODE) <= 3 * rem + 2;
            const int lev = (int)(wp & 63u), slot = (int)(wp >> PATH_SLOT) & 0xff;
            const uint32_t pe = act ? L.pend[slot] : END_SKIP;
            const int li = (int)(pe & 0x3ffu), lj = (int)(pe >> 10) & 0x3ff;
            R qq = zero;
            if (!(pe & END_SKIP)) {
                const size_t np = (size_t)P.nblk * T;
                const double* pc = P.pconst + (size_t)b * T + l;
                PathEnds<R> pn;
                pn.ri_d = pc[0]; pn.rj_d = pc[np];
                pn.di = L.dph[li]; pn.dj = L.dph[lj];
                pn.dpi = L.dphp[li]; pn.dpj = L.dphp[lj];
                if (LEV) {
                    pn.lev_i = pe & END_LEV_I; pn.lev_j = pe & END_LEV_J;
                    if (pn.lev_i) { pn.ldi = L.ldph[li]; pn.ei = M.elevtn[M.pth_upst[gp]]; }
                    if (pn.lev_j) { pn.ldj = L.ldph[lj]; pn.ej = M.elevtn[M.pth_down[gp]]; }
                }
                const R before = pf;
                qq = path_level<R>(pn, path_slope<R>(pn, R(pc[4 * np])), LEV, lev, pc[2 * np], R(gdt), [&](R& w, R& man, R& pre) {
                    w = R(pc[3 * np]);
                    man = R(M.pth_man[lev]);
                    pre = before;
                });
            }
            R sum = zero;
            const int lane = l & 63, base = lane - lev;
            for (int k = 0; k < M.npthlev; ++k) sum = sum + __shfl(qq, base + k);
            if (act) {
                if (sum != zero) {                                        // pthout:84-95
                    R rate = (R(0.05) * vmin(L.sto[li], L.sto[lj])) / vabs(sum * R(dt));
                    rate = vmin(rate, R(1));
                    qq = qq * rate;
                    sum = sum * rate;
                }
                pf = qq;
                if (lev == 0) L.psum[slot] = sum;
            }
        }
        // ---- outflow (k_outflow)
        if (code <= 3 * rem + 2) {
            FlowIn<R> c;
            c.rivdph = L.dph[l]; c.rivdph_pre = L.dphp[l];
            c.qr_pre = ro;
            c.qr_old = it == 0 && a.vel0 ? a.vel0[s0] : c.qr_pre;
            c.fldsto = R(fs); c.flddph = L.fdph[l]; c.fldsto_pre = L.fpre[l];
            c.fldout_pre = fo;
            double stg = rs + fs;
            if (is_lev) stg = stg + L.lev[l];
            c.storge = R(stg);
            c.elevtn = f_elevtn; c.rivhgt = f_rivhgt; c.rivwth = f_rivwth; c.rivman = f_rivman;
            c.nxtdst = f_nxtdst; c.rivlen = f_rivlen;
            c.river = river;
            c.dj = river ? L.dph[nx] : zero;
            c.dj_pre = river ? L.dphp[nx] : zero;
            c.zdn = zdn;
            const Surface<R> sf = surface_of<R>(c);
            R q_r, q_f, vel = river_vel<R>(c, sf);
            const int bits = is_dam ? L.dcode[e] : 0;
            if (!DAM || !(bits & DAM_CODE)) {
                local_inertial<R>(c, sf, A.lfldout, A.pmanfld, A.pdstmth, dt, gdt, q_r, q_f);
            } else {
                const BlockArgs<R>& ad = block_args<R>();
                double inf = (double)ad.S.runoff[s0];                      // damout:447-464
                const int nd = ad.P.ndam[b];
                for (int k = 0; k < nup; ++k) {
                    const int u = k == 0 ? u0 : (k == 1 ? u1 : (int)ad.P.upx[ad.P.upx_ptr[b * T + l] + k - 2]);
                    const bool dam_up = u < (nd & 0xffff) || (u >= BLK_KINE_AT && u < BLK_KINE_AT + (nd >> 16));
                    const int eu = dam_up ? slot_of_dam(u, T) : 0;
                    const int cu = dam_up ? L.dcode[eu] & DAM_CODE : 0;
                    if (cu == 10 || cu == 11) inf = (inf + (double)L.ro[eu]) + (double)L.fo[eu];
                }
                L.daminf[e] = inf;
                dam_outflow<R>(ad.M, (bits & DAM_KINE) != 0, L.vk[e], L.vf[e], f_rivwth, f_rivlen,
                               (bits & DAM_ACTIVE) != 0, L.drow[e], inf, dt, L.dph[l], L.fdph[l], rs, fs, L.dam[e],
                               q_r, q_f, vel);
            }
            L.q[l] = q_r;
            L.f[l] = q_f;
            if (own) {
                if (last) S.rivvel[s0] = vel;
                L.a_vel[l] = L.a_vel[l] + vel * rdt;
            }
        }
        sync_lds();
        const bool upd = code <= 3 * rem;
        const R runoff = upd ? S.runoff[s0] : zero;                        // in flight during the rate phase
        const int npo = PTH ? (int)(wc >> 16) & 0xff : 0, npa = PTH ? npo + (int)(wc >> 24) : 0;
        R pavg = zero, qavg = zero;                                       // as these
        const bool pupd = PTH && gp >= 0 && (int)(wp >> PATH_CODE) <= 3 * rem, pown = pupd && (wp >> PATH_CODE) == 0;
        if (PTH && it > 0) {
            if (own && npa > 0) pavg = S.pthout_avg[s0];
            if (pown) qavg = S.pthflw_avg[(size_t)(wp & 63u) * M.nsp + gp];
        }
        auto slot_at = [&](int k) {
            return k == 0 ? (int)(wc & 0xffu) : (k == 1 ? (int)(wc >> 8) & 0xff : (int)P.ppx[P.ppx_ptr[b * T + l] + k - 2]);
        };
        // ---- limiter rate (k_rate)
        if (code <= 3 * rem + 1) {
            double so = (double)vmax(L.q[l], zero) + (double)vmax(L.f[l], zero);
            if (nup > 0) so = (so + (double)vmax(-L.q[u0], zero)) + (double)vmax(-L.f[u0], zero);
            if (nup > 1) so = (so + (double)vmax(-L.q[u1], zero)) + (double)vmax(-L.f[u1], zero);
            for (int k = 2; k < nup; ++k) {
                const int u = P.upx[P.upx_ptr[b * T + l] + k - 2];
                so = (so + (double)vmax(-L.q[u], zero)) + (double)vmax(-L.f[u], zero);
            }
            so = so * dt;
            for (int k = 0; k < npa; ++k) {
                const R v = L.psum[slot_at(k)];
                so = so + (double)vmax(k < npo ? v : -v, zero) * dt;
            }
            const R dout = vmax(R(so), R(1.e-10));
            L.rate[l] = vmin(R(rs + fs) / dout, R(1));
        }
        sync_lds();
        // a path's sum under the rate of the end it leaves
        auto limited = [&](R v, uint32_t pe) {
            return pe & END_NOLIM ? v : (v >= zero ? v * L.rate[pe & 0x3ffu] : v * L.rate[(pe >> 10) & 0x3ffu]);
        };
        if (PTH && pupd) {                                                // update_path
            const int lev = (int)(wp & 63u);
            pf = limited(pf, L.pend[(wp >> PATH_SLOT) & 0xffu]);
            if (pown) {
                qavg = qavg + pf * rdt;
                if (last) qavg = qavg / R(a.I.nadd);
                S.pthflw_avg[(size_t)lev * M.nsp + gp] = qavg;
            }
        }
        if (PTH && last && __any(pown)) {
            const int lev = (int)(wp & 63u), slot = (int)(wp >> PATH_SLOT) & 0xff, base = (l & 63) - lev;
            R sumavg = zero;                                              // diag:206-213
            for (int k = 0; k < M.npthlev; ++k) sumavg = sumavg + __shfl(qavg, base + k);
            if (pown && lev == 0) {
                S.pthflwsum[gp] = limited(L.psum[slot], L.pend[slot]);
                S.pthflwsum_avg[gp] = sumavg;
            }
        }
        // ---- limit, inflow, dam balance, storages (k_update)
        {
            double gb[NGLB];
#pragma unroll
            for (int k = 0; k < NGLB; ++k) gb[k] = 0.0;
            if (upd) {
                const R qr = L.q[l], qf = L.f[l], ri = L.rate[l];
                const R r = (river && !(qr > zero)) ? L.rate[nx] : ri;
                const R qrl = qr * r, qfl = qf * r;
                double rivinf = 0.0, fldinf = 0.0;
                auto inflow = [&](int u) {
                    const R qu = L.q[u], fu = L.f[u];
                    const R ru = (qu > zero) ? L.rate[u] : ri;
                    rivinf = rivinf + (double)(qu * ru);
                    fldinf = fldinf + (double)(fu * ru);
                };
                if (nup > 0) inflow(u0);
                if (nup > 1) inflow(u1);
                for (int k = 2; k < nup; ++k) inflow(P.upx[P.upx_ptr[b * T + l] + k - 2]);
                double pthout = 0.0;
                for (int k = 0; k < npa; ++k) {                           // inflow_lspamat:519-535
                    const int sl = slot_at(k);
                    const double v = (double)limited(L.psum[sl], L.pend[sl]);
                    pthout = k < npo ? pthout + v : pthout - v;
                }
                if (is_dam && (L.dcode[e] & DAM_BALANCE))
                    L.dam[e] = (L.dam[e] + ((rivinf + fldinf) + (double)runoff) * dt) - ((double)qrl + (double)qfl) * dt;
                L.fpre[l] = R(fs);
                const R outflw = qrl + qfl;
                storage_next<R>(rs, fs, rivinf, fldinf, pthout, qrl, qfl, dt, runoff, L.ffrc[l], A.lupsinf,
                                A.lupsinf ? S.upsinf[s0] : zero, gb);
                double st = rs + fs;
                if (is_lev) st = st + L.lev[l];
                gb[G_STONEW] = (double)R(st);
                gb[G_STOPRE2] = st;
                ro = qrl; fo = qfl;
                if (is_dam) { L.ro[e] = qrl; L.fo[e] = qfl; }
                if (own) {
                    L.a_riv[l] = L.a_riv[l] + qrl * rdt;
                    L.a_fld[l] = L.a_fld[l] + qfl * rdt;
                    if (!kOutSum) L.a_out[l] = L.a_out[l] + outflw * rdt;
                    L.m_out[l] = vmax(L.m_out[l], vabs(outflw));
                    if (is_dam) L.a_inf[e] = L.a_inf[e] + R(L.daminf[e] * dt);
                    if (PTH && npa > 0) {
                        R pa = pavg + R(pthout) * rdt;
                        if (last) pa = pa / R(a.I.nadd);
                        S.pthout_avg[s0] = pa;
                    }
                    if (last) {
                        S.rivinf[s0] = rivinf; S.fldinf[s0] = fldinf; S.pthout[s0] = pthout;
                        S.outflw[s0] = outflw;
                    }
                }
            }
            if (!MB && A.budget) {
                double ga[NA];
#pragma unroll
                for (int k = 0; k < NA; ++k) ga[k] = own ? gb[k] : 0.0;      // the owner counts a cell
                wave_sum_comp<NA>(ga, L.sum, L.sum + NGLB * NW, NW, l >> 6);
            }
        }
        // ---- stage inversion, maxima
        {
            double gs[NB];
#pragma unroll
            for (int k = 0; k < NB; ++k) gs[k] = 0.0;
            if (upd) {
                Stage o;
                const Geom geo{(double)f_rivlen, (double)f_rivwth, (double)f_grarea, (double)f_rivhgt};
                using Lds = BlockLds<R, T, LEV, DAM, PTH>;
                const BlockHgt<Lds::NL, T> hgt{&L.hgt[0][l], M.fldhgt + g, M.n};
                if (is_lev) stage_levee(M, hgt, geo, load_lev_row(M, L.lrow[l]), rs, fs, L.lev[l], o);
                else stage_def<!LEV>(M, hgt, geo, rs, fs, o);
                rs = o.rivsto;
                fs = o.fldsto;
                double stg = rs + fs;
                if (is_lev) L.lev[l] = o.levsto;
                if (LEV) stg = stg + o.levsto;
                const R rivdph = R(o.rivdph), storge = R(stg);
                L.dphp[l] = L.dph[l];
                L.dph[l] = rivdph;
                L.fdph[l] = R(o.flddph);
                L.ffrc[l] = R(o.fldfrc);
                if (PTH) {
                    L.sto[l] = storge;
                    if (is_lev) L.ldph[l] = R(o.levdph);
                }
                if (own) {
                    gs[0] = stg;
                    gs[G_RIVSTO - G_STONEW2] = rs;
                    gs[G_FLDSTO - G_STONEW2] = fs;
                    gs[G_FLDARE - G_STONEW2] = o.fldare;
                    if (LEV) gs[NB - 1] = o.levsto;
                    L.m_dph[l] = vmax(L.m_dph[l], rivdph);
                    L.m_sto[l] = vmax(L.m_sto[l], storge);
                    if (last) {
                        S.fldare[s0] = R(o.fldare);
                        S.sfcelv[s0] = R((double)f_elevtn - (double)f_rivhgt) + rivdph;
                        S.storge[s0] = storge;
                        if (!PTH && is_lev) S.levdph[s0] = R(o.levdph);
                    }
                }
            }
            if (!MB && A.budget) wave_sum_comp<NB>(gs, L.sum, L.sum + NGLB * NW, NW, l >> 6, G_STONEW2);
        }
        sync_lds();
        // the wavefront sums stay until the next update, two barriers from here
        if (!MB && A.budget && l < NGLB) {
            const int k = l == G_STOPRE2 && !kOutSum ? (int)G_STONEW : l;
            double hi = 0.0, lo = 0.0;
            if (LEV || k != G_LEVSTO) comp_total(L.sum, L.sum + NGLB * NW, NW, k, hi, lo);
            double* part = S.partials + ((size_t)it * P.nblk + b) * NPART;
            part[l] = hi;
            part[NGLB + l] = lo;
        }
    }
    if (PTH && gp >= 0 && (wp >> PATH_CODE) == 0) {
        const BlockArgs<R>& a = block_args<R>();
        a.O.pthflw[(size_t)(wp & 63u) * a.M.nsp + gp] = pf;
    }
    if (g < 0 || (w1 >> TOPO_CODE) != 0) return;
    const BlockArgs<R>& a = block_args<R>();
    const DevState<R>& S = a.S;
    const BlockState<R>& O = a.O;
    const R rdt = R(dt);
    O.rivsto[s0] = rs; O.fldsto[s0] = fs;
    O.rivout[s0] = ro; O.fldout[s0] = fo;
    O.rivdph[s0] = L.dph[l]; O.rivdph_pre[s0] = L.dphp[l];
    O.fldsto_pre[s0] = L.fpre[l]; O.flddph[s0] = L.fdph[l]; O.fldfrc[s0] = L.ffrc[l];
    if (LEV && (w0 & (BLK_LEV << TOPO_FLAGS))) {
        O.levsto[s0] = L.lev[l];
        if (PTH) O.levdph[s0] = L.ldph[l];
    }
    const bool is_dam = DAM && (w0 & (BLK_DAM << TOPO_FLAGS));
    const int e = slot_of_dam(l, T);
    if (is_dam) { O.damsto[s0] = L.dam[e]; S.daminf[s0] = L.daminf[e]; }
    R a4 = is_dam ? L.a_inf[e] : zero;                                     // daminf_sparse: zero elsewhere
    S.outflw_max[s0] = L.m_out[l]; S.rivdph_max[s0] = L.m_dph[l]; S.storge_max[s0] = L.m_sto[l];
    R a1 = L.a_riv[l], a2 = L.a_fld[l], av = L.a_vel[l], a3 = kOutSum ? zero : L.a_out[l];
    if (it0 + nsub == nt) {                                               // GETAVE, diag:179-186
        const R nadd = R(MB ? S.inst[(a.P.dom[b] << a.M.lgm) + m].nadd : a.I.nadd);
        a1 = a1 / nadd; a2 = a2 / nadd; av = av / nadd;
        a3 = kOutSum ? a1 + a2 : a3 / nadd;
        const R runoff = S.runoff[s0];
        R a5 = zero;
        for (int k = 0; k < nt; ++k) a5 = a5 + runoff * rdt;
        S.runoff_avg[s0] = a5 / nadd;
        if (!PTH || (wc >> 16) == 0) S.pthout_avg[s0] = zero;
        a4 = a4 / nadd;
        S.outflw_avg[s0] = a3;
    } else if (!kOutSum) {
        S.outflw_avg[s0] = a3;
    }
    if (is_dam || (DAM && it0 + nsub == nt)) S.daminf_avg[s0] = a4;
    S.rivout_avg[s0] = a1; S.fldout_avg[s0] = a2; S.rivvel_avg[s0] = av;
}

template <class R, int T, bool MB, bool PTH>
static hipError_t launch_block_t(const BlockArgs<R>& a, hipStream_t st) {
    const dim3 g(((a.P.nblk + 7) / 8 * 8) << (MB ? a.M.lgm : 0)), t(T);
    if (a.A.llevee && a.A.ldamout) hipLaunchKernelGGL((k_block<R, T, true, true, MB, PTH>), g, t, 0, st, a);
    else if (a.A.llevee) hipLaunchKernelGGL((k_block<R, T, true, false, MB, PTH>), g, t, 0, st, a);
    else if (a.A.ldamout) hipLaunchKernelGGL((k_block<R, T, false, true, MB, PTH>), g, t, 0, st, a);
    else hipLaunchKernelGGL((k_block<R, T, false, false, MB, PTH>), g, t, 0, st, a);
    return hipGetLastError();
}

template <class R, bool MB>
static hipError_t launch_block_mb(const BlockArgs<R>& a, hipStream_t st) {
    switch (a.P.T) {
        case 256: return launch_block_t<R, 256, MB, false>(a, st);
        case 512: return launch_block_t<R, 512, MB, false>(a, st);
        default: return launch_block_t<R, 1024, MB, false>(a, st);
    }
}

// flows of the paths with an end outside the network, which no block holds (update_path)
template <class R>
__global__ void k_dead_paths(DevMap M, DevState<R> S, const int32_t* dead, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int q = dead[k];
    for (int l = 0; l < M.npthlev; ++l) {
        S.pthflw[(size_t)l * M.nsp + q] = R(0);
        S.pthflw_avg[(size_t)l * M.nsp + q] = R(0);
    }
    S.pthflwsum[q] = R(0);
    S.pthflwsum_avg[q] = R(0);
}

template <class R>
hipError_t launch_block(const DevMap& M, const DevState<R>& S, const BlockState<R>& O, const BlockTab& P,
                        const StepArgs& A, const InstStep& I, int j, const R* vel0, hipStream_t st) {
    const BlockArgs<R> a{M, S, O, P, A, I, j, vel0};
    if (j == 0 && P.ndead > 0)                                       // also where every path is dead
        hipLaunchKernelGGL((k_dead_paths<R>), dim3((P.ndead + 255) / 256), dim3(256), 0, st, M, S, P.dead, P.ndead);
    if (P.npth > 0) {
        switch (P.T) {
            case 256: return launch_block_t<R, 256, false, true>(a, st);
            default: return launch_block_t<R, 512, false, true>(a, st);
        }
    }
    if (M.nmem > 1 || M.cell_dom) return launch_block_mb<R, true>(a, st);
    return launch_block_mb<R, false>(a, st);
}
template hipError_t launch_block<double>(const DevMap&, const DevState<double>&, const BlockState<double>&,
                                         const BlockTab&, const StepArgs&, const InstStep&, int, const double*,
                                         hipStream_t);
template hipError_t launch_block<float>(const DevMap&, const DevState<float>&, const BlockState<float>&,
                                        const BlockTab&, const StepArgs&, const InstStep&, int, const float*,
                                        hipStream_t);

}  // namespace cmf
