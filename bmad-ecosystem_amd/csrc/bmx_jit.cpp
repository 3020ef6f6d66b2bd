// Lattice-specialised tile kernels, compiled at run time.
//
// A ring is mostly one cell repeated: the same element kinds and flags in the same order, with
// parameter blocks of the same size. For such a lattice the element loop of the tile kernel
// can be written out once per cell position with the kind and flags as compile-time constants:
// every kind dispatch and flag test folds away, and each map's results flow straight into the
// next element's code instead of through the joins of a dispatch. The source of that turn
// policy is generated here, compiled with hiprtc for the device together with the library's
// own device headers (embedded at build time, bmx_jit_sources.cpp), and loaded as a module.
// Elements outside the repeated run (a head cell that differs, the tail with the rf cavity)
// keep the generic table-driven loop. Kernels are cached per device and cell signature, so
// lattices that differ only in element strengths (error variants) share one.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "bmx_internal.hpp"

extern const char bmx_jit_src_table[];
extern const char bmx_jit_src_maps[];
extern const char bmx_jit_src_fast[];
extern const char bmx_jit_src_tiles[];

namespace bmx {

struct JitKernels {
    hipModule_t module = nullptr;
    hipFunction_t fn[3] = {};  // waves per SIMD 3, 4, 5
    bool rare_q = false;       // carries K_QMULT / K_BMULT on its rare path (all built for 2 waves)
    int level = 0;             // 0 plain, 1 stepped elements, 2 with radiation kicks
};

namespace {

// head elements [0, H) generic, then N cells of P elements, cell c's parameters at
// hdr[H].off + c * S, then the tail generic.
struct Period {
    int32_t H = 0, P = 0, N = 0, S = 0;
};

bool cell_repeats(const HostTable &t, int32_t H, int32_t P, int32_t N, int32_t S)
{
    for (int32_t c = 1; c < N; c++)
        for (int32_t j = 0; j < P; j++) {
            const EleHdr &a = t.hdr[H + j], &b = t.hdr[H + c * P + j];
            if (a.kind != b.kind || a.flags != b.flags || a.n != b.n || b.off != a.off + c * S)
                return false;
        }
    return true;
}

// The shortest cell (up to 64 elements) that repeats over at least three quarters of the
// lattice, starting at element 0 or after one differing head cell.
bool find_period(const HostTable &t, Period &out)
{
    const int32_t n = (int32_t)t.hdr.size();
    for (int32_t P = 1; P <= 64 && 4 * P <= n; P++) {
        for (int32_t H : {0, P}) {
            if (H + 2 * P > n) continue;
            const int32_t S = t.hdr[H + P].off - t.hdr[H].off;
            int32_t N = 1;
            while (H + (N + 1) * P <= n && cell_repeats(t, H, P, N + 1, S)) N++;
            if (N >= 4 && 4 * N * P >= 3 * n) {
                out = {H, P, N, S};
                return true;
            }
        }
    }
    return false;
}

// How the cell kernels track the element at a cell position: on its operations where every cell has
// the same ones there (their tests on entering united), by the general maps written out where no cell has
// any, and by the tables where the cells differ.
enum CellForm : char { CELL_GENERAL = 0, CELL_OPS = 1, CELL_TABLE = 2 };
CellForm cell_ops(const HostTable &t, const Period &pd, int32_t j, std::vector<uint32_t> &codes, bool &open)
{
    open = false;
    const int32_t n = t.fast[pd.H + j].n_ops;
    codes.assign(n, 0);
    for (int32_t c = 0; c < pd.N; c++) {
        const int32_t i = pd.H + c * pd.P + j;
        const FastEle &fe = t.fast[i];
        if (fe.n_ops != n) return CELL_TABLE;
        open |= t.fast_open[i] != 0;
        for (int32_t k = 0; k < n; k++) {
            const uint32_t v = (uint32_t)(fe.codes[k >> 3] >> (8 * (k & 7)) & 255);
            if (c > 0 && (v & ~FO_UCHECK) != (codes[k] & ~FO_UCHECK)) return CELL_TABLE;
            codes[k] |= v;
        }
    }
    return n > 0 ? CELL_OPS : CELL_GENERAL;
}

// The coefficients of a radiation kick that are not zero in some cell: damp_dmat[i][j] in bit
// 6 i + j, xfer_damp_vec[i] in bit 36 + i, stoc_mat's lower triangle by rows, and the masks of
// rows and columns that fast_radiation's packed word has, which must be the same in every cell.
// The kick's values in the stream: that word, ref_orb of the columns of damp_dmat in use, each
// damping row's coefficients and xfer_damp_vec, each stochastic row's coefficients. Read row by
// row from the packed map (fast_radiation), a kick of the usual bend waits for 8 lines one after
// the other; these values are 24, and come with the cell's.
struct RadTerms {
    uint64_t damp = 0;
    uint32_t stoc = 0, cols = 0;
    bool energy = false;
    bool columns(int j) const { return damp & (0x041041041ull << j) & 0xFFFFFFFFFull; }
};

// Where the values of a cell's operations lie in its stream (LatDesc::cell): lines of kFastOpLen
// doubles, an operation's values within one line (they are in scalar registers together, and
// the next line is loaded while the operations of one run). An aperture equal to the one before
// in every cell is kept, not stored again.
struct CellOp {
    int32_t j, k;        // element of the cell, operation of the element
    uint32_t code;
    int32_t at;          // first value in the stream
    int32_t ap;          // its aperture's k2 in the stream (r2 next), or -1: none
    int32_t n = 0;       // its values
    RadTerms rad;        // a radiation kick written out
};
struct CellPlan {
    std::vector<CellOp> ops;
    std::vector<char> fast, open;  // per element: CellForm; its last operation leaves px, py untested
    int32_t lines = 0;
};

const double *op_record(const HostTable &t, const Period &pd, int32_t c, const CellOp &o)
{
    return &t.ops[(size_t)kFastOpLen * (t.fast[pd.H + c * pd.P + o.j].op0 + o.k)];
}

// The packed word of a radiation kick, and its map's values line by line in the order of RadTerms.
uint64_t rad_word(const double *record)
{
    uint64_t at;
    std::memcpy(&at, record, sizeof at);
    return at;
}

struct RadMap {
    double ref[6] = {}, damp[6][6] = {}, xfer[6] = {}, stoc[6][6] = {};
};

RadMap rad_map(const HostTable &t, uint64_t at)
{
    RadMap m;
    const double *l = &t.rad_lines[(size_t)kFastOpLen * (at & 0xFFFFFF)];
    std::copy(l, l + 6, m.ref);
    for (int i = 0; i < 6; i++)
        if (at >> (26 + i) & 1) {
            l += kFastOpLen;
            std::copy(l, l + 6, m.damp[i]);
            m.xfer[i] = l[6];
        }
    for (int i = 0; i < 6; i++)
        if (at >> (32 + i) & 1) {
            l += kFastOpLen;
            std::copy(l, l + i + 1, m.stoc[i]);
        }
    return m;
}

// The terms of a kick that is one in every cell with the same rows and columns; else none (n = 0).
int32_t rad_terms(const HostTable &t, const Period &pd, const CellOp &o, RadTerms &r)
{
    const uint64_t masks = rad_word(op_record(t, pd, 0, o)) >> 24 & 0xFFFFF;  // edge, rows, columns
    for (int32_t c = 0; c < pd.N; c++) {
        const uint64_t at = rad_word(op_record(t, pd, c, o));
        if ((at >> 24 & 0xFFFFF) != masks) return 0;
        const RadMap m = rad_map(t, at);
        for (int i = 0, k = 0; i < 6; i++) {
            for (int j = 0; j < 6; j++)
                if (m.damp[i][j] != 0) r.damp |= 1ull << (6 * i + j);
            if (m.xfer[i] != 0) r.damp |= 1ull << (36 + i);
            for (int j = 0; j <= i; j++, k++)
                if (m.stoc[i][j] != 0) r.stoc |= 1u << k;
        }
    }
    r.cols = masks >> 14 & 63;
    r.energy = ((masks >> 2 | masks >> 8) >> 5) & 1;
    int32_t n = 1 + __builtin_popcountll(r.damp) + __builtin_popcount(r.stoc);
    for (int j = 0; j < 6; j++) n += r.columns(j);
    return n;
}

// The values of an operation of cell c in the order of its places in the stream.
std::vector<double> op_values(const HostTable &t, const Period &pd, int32_t c, const CellOp &o)
{
    const double *r = op_record(t, pd, c, o);
    if (!o.rad.cols && !o.rad.damp) return std::vector<double>(r, r + o.n);
    std::vector<double> v{r[0]};
    const RadMap m = rad_map(t, rad_word(r));
    for (int j = 0; j < 6; j++)
        if (o.rad.columns(j)) v.push_back(m.ref[j]);
    for (int i = 0; i < 6; i++) {
        for (int j = 0; j < 6; j++)
            if (o.rad.damp >> (6 * i + j) & 1) v.push_back(m.damp[i][j]);
        if (o.rad.damp >> (36 + i) & 1) v.push_back(m.xfer[i]);
    }
    for (int i = 0, k = 0; i < 6; i++)
        for (int j = 0; j <= i; j++, k++)
            if (o.rad.stoc >> k & 1) v.push_back(m.stoc[i][j]);
    return v;
}

CellPlan plan_cell(const HostTable &t, const Period &pd)
{
    CellPlan p;
    p.fast.assign(pd.P, 0);
    p.open.assign(pd.P, 0);
    int32_t at = 0, ap = -1;
    CellOp last{};
    auto place = [&](int32_t n) {  // n values within one line
        if (at % kFastOpLen + n > kFastOpLen) at += kFastOpLen - at % kFastOpLen;
        const int32_t r = at;
        at += n;
        return r;
    };
    for (int32_t j = 0; j < pd.P; j++) {
        std::vector<uint32_t> codes;
        bool open;
        p.fast[j] = cell_ops(t, pd, j, codes, open);
        if (p.fast[j] != CELL_OPS) {
            ap = -1;
            continue;
        }
        p.open[j] = open;
        for (size_t k = 0; k < codes.size(); k++) {
            CellOp o{j, (int32_t)k, codes[k], 0, -1};
            const uint32_t kind = codes[k] & FO_KIND;
            if (!fast_untested(kind)) {
                bool same = ap >= 0;
                for (int32_t c = 0; c < pd.N && same; c++) {
                    const double *a = op_record(t, pd, c, o), *b = op_record(t, pd, c, last);
                    same = a[6] == b[6] && a[7] == b[7];
                }
                if (!same) ap = place(2);
                o.ap = ap;
                last = o;
            }
            o.n = kind == FO_RAD ? rad_terms(t, pd, o, o.rad) : 0;
            if (o.n > 1) {  // taken one by one, over the ends of lines
                o.at = at;
                at += o.n;
            } else {
                o.rad = RadTerms{};
                o.n = fast_values(kind);
                o.at = place(o.n);
            }
            p.ops.push_back(o);
        }
    }
    p.lines = (at + kFastOpLen - 1) / kFastOpLen;
    if (p.lines == 1) p.lines = 2;  // a line is loaded while the one before is in use
    return p;
}

// A radiation kick on the terms of its maps that are not zero (the arithmetic of fast_radiation with
// the zero terms left out), each value taken as the stream brings it.
template <class Reach, class Val>
void write_radiation(std::ostream &b, const CellOp &o, size_t id, Reach &reach, Val &val)
{
    int32_t at = o.at;
    const auto next = [&]() {
        reach(at);
        return val(at++);
    };
    const std::string k = std::to_string(id), in = "                ";
    const std::string word = next();
    if (o.code & FO_UCHECK) b << in << "fast_unstable(f, ef, bad);\n";
    b << in << "const uint64_t at" << k << " = __double_as_longlong(" << word << ");\n"
      << in << "double g" << k << "[6] = {0, 0, 0, 0, 0, 0};\n"
      << in << "if (L.sp.rad.flags & RAD_FLUCT) rad_deviates(g" << k << ", at" << k << ", " << o.rad.cols
      << "u, L.sp, ra);\n"
      << in << "bad |= lanes(!(fabs(f.z) < 1e30));\n"
      << in << "double v" << k << "[6] = {f.x, f.px, f.y, f.py, f.z, ef.pz};\n"
      << in << "double d" << k << "[6] = {0, 0, 0, 0, 0, 0}, s" << k << ";\n";
    for (int j = 0; j < 6; j++)
        if (o.rad.columns(j)) {
            const std::string v = next();
            b << in << "d" << k << "[" << j << "] = v" << k << "[" << j << "] - " << v << ";\n";
        }
    // a row's sum over its terms, then coordinate i moved by it where `when` holds
    const auto row = [&](int i, int n, uint64_t mask, const char *x, const char *when) {
        bool any = false;
        for (int j = 0; j < n; j++) {
            if (!(mask >> j & 1)) continue;
            const std::string c = next(), xj = x + k + "[" + std::to_string(j) + "]";
            if (any) b << in << "s" << k << " = fma(" << c << ", " << xj << ", s" << k << ");\n";
            else b << in << "s" << k << " = " << c << " * " << xj << ";\n";
            any = true;
        }
        const std::string vi = "v" + k + "[" + std::to_string(i) + "]";
        if (any) b << in << "if (" << when << ") " << vi << " = fma(L.sp.rad.scale, s" << k << ", " << vi << ");\n";
    };
    for (int i = 0; i < 6; i++) {
        row(i, 6, o.rad.damp >> (6 * i) & 63, "d", "L.sp.rad.flags & RAD_DAMP");
        if (o.rad.damp >> (36 + i) & 1) {
            const std::string x = next(), vi = "v" + k + "[" + std::to_string(i) + "]";
            b << in << "if ((L.sp.rad.flags & (RAD_DAMP | RAD_ZERO_AVERAGE)) == RAD_DAMP) " << vi
              << " = fma(L.sp.rad.scale, " << x << ", " << vi << ");\n";
        }
    }
    for (int i = 0, t = 0; i < 6; t += ++i) row(i, i + 1, o.rad.stoc >> t & ((1u << (i + 1)) - 1), "g", "L.sp.rad.flags & RAD_FLUCT");
    b << in << "rad_leave(f, ef, v" << k << ", " << (o.rad.energy ? "true" : "false") << ", L.sp, bad);\n";
}

// The map set the cell kernels of a lattice carry on their rare path, by all its elements: those of
// the head and the tail are tracked by these kernels too.
struct CellMaps {
    bool q_kinds = false;  // stepped quadrupoles or general bends
    const char *rare;
};

CellMaps cell_maps(const HostTable &t)
{
    CellMaps m;
    for (const EleHdr &h : t.hdr) m.q_kinds |= h.kind == K_QMULT || h.kind == K_BMULT;
    m.rare = t.rad ? (m.q_kinds ? "MAPS_RARE_QR" : "MAPS_RARE_R") : t.rare_q ? "MAPS_RARE_Q" : "MAPS_RARE";
    return m;
}

// All that the kernels' source is made from, and so their key in the cache. Taken without writing
// the source, which a lattice whose kernels are there does not need.
std::string signature(const HostTable &t, const Period &pd, const CellPlan &plan, const CellMaps &maps)
{
    std::string key = maps.rare;
    const auto put = [&](auto v) { key.append((const char *)&v, sizeof v); };
    for (const int32_t v : {pd.H, pd.P, pd.N, pd.S, (int32_t)t.hdr.size(), t.hdr[pd.H].off, (int32_t)maps.q_kinds}) put(v);
    for (int32_t j = 0; j < pd.P; j++) {
        const EleHdr &h = t.hdr[pd.H + j];
        for (const int32_t v : {h.kind, h.flags, h.n, h.off - t.hdr[pd.H].off}) put(v);
        put(plan.fast[j]);
        put(plan.open[j]);
    }
    for (const CellOp &o : plan.ops) {
        for (const int32_t v : {o.j, o.k, (int32_t)o.code, o.at, o.ap, o.n}) put(v);
        put(o.rad.damp);
        put(o.rad.stoc);
        put(o.rad.cols);
        put(o.rad.energy);
    }
    return key;
}

std::string generate(const HostTable &t, const Period &pd, const CellPlan &plan, const CellMaps &maps)
{
    std::ostringstream body;
    // The cell in segments: runs of at most kFastBlockOps operations (bmx_fast.hpp), and its other
    // elements, whose general maps are written out with their kinds and flags as constants. A run that
    // refuses lanes leaves the cell loop with its element range and the next segment's
    // number; the table-driven loop's one call site takes them through the range and the cell
    // loop is entered again there. Lanes that an element of the general maps loses leave it too.
    // (Left to the table-driven loop as well, those elements took 1.3 to 2.5 times as long: a
    // stepped quadrupole in each cell, 100000 particles, 200 elements, 3 turns 1555 us against
    // 473, octupoles 801 against 342, bends beyond 0.1 rad 872 against 495.)
    size_t next_op = 0;
    // A cell with such elements also keeps a wave with a lane near the zero orbit, which a cell of
    // operations alone leaves to the tables: its runs have the semi-linear bend.
    const bool mixed = std::count(plan.fast.begin(), plan.fast.end(), CELL_GENERAL) > 0;
    // One run that is the whole cell loads the next cell's first line behind its last one and
    // carries it over; otherwise each run loads its own first line.
    bool carry = (int32_t)plan.ops.size() <= kFastBlockOps && !plan.ops.empty();
    for (int32_t j = 0; j < pd.P; j++) carry = carry && plan.fast[j] == CELL_OPS;
    int32_t n_seg = 0;
    auto leave = [&](int32_t j0, int32_t j1) {
        std::ostringstream r;
        r << "e0 = eb + " << j0 << "; e1 = eb + " << j1 << "; ";
        if (j1 == pd.P) r << "seg = 0; ++c; break;";
        else r << "seg = " << n_seg + 1 << "; break;";
        return r.str();
    };
    for (int32_t j = 0; j < pd.P;) {
        body << "            case " << n_seg << ":\n";
        if (plan.fast[j] == CELL_GENERAL) {
            int32_t j1 = j;
            bool energy = false;
            for (; j1 < pd.P && plan.fast[j1] == CELL_GENERAL; j1++) {
                const EleHdr &h = t.hdr[pd.H + j1];
                // the rare set where the table-driven loops take it; elsewhere pz cannot change
                const bool rare = h.kind == K_RF || (h.flags & (F_OFFSET | F_APE_MOMENTUM | F_RARE_MAP));
                energy |= rare;
                body << "                if (p.state == ST_ALIVE)\n"
                     << "                    track_element<true, " << (rare ? "kRare" : "MAPS_NO_RF") << ">(p, EleRef{" << h.kind
                     << ", " << h.flags << ", " << h.n << ", " << h.off - t.hdr[pd.H].off << "}, base, L.sp, true, eb + "
                     << j1 + 1 << ", t_abs);\n";
            }
            if (energy)
                body << "                en = fast_energy(p, L.sp);\n"
                     << "                near = !maps_rad(kRare) && near_zero<kRare>(p);\n";
            body << "                who = lanes(p.state != ST_ALIVE);\n"
                 << "                if (who) { " << leave(j1, j1) << " }\n";
            n_seg++;
            j = j1;
            continue;
        }
        if (plan.fast[j] == CELL_TABLE) {
            int32_t j1 = j + 1;
            while (j1 < pd.P && plan.fast[j1] == CELL_TABLE) j1++;
            body << "                who = ~(LaneMask)0;\n                " << leave(j, j1) << '\n';
            n_seg++;
            j = j1;
            continue;
        }
        // elements [j, j1) in one run
        int32_t j1 = j, n = 0;
        size_t o1 = next_op;
        bool open = false;
        while (j1 < pd.P && plan.fast[j1] == CELL_OPS) {
            size_t o = o1;
            while (o < plan.ops.size() && plan.ops[o].j == j1) o++;
            if (n > 0 && n + (int32_t)(o - o1) > kFastBlockOps) break;
            n += (int32_t)(o - o1);
            if (o > o1) open = plan.open[j1];
            o1 = o;
            j1++;
        }
        if (n > 0) {
            // the lines the run reads
            int32_t first_line = INT32_MAX, last_line = -1, ap = -1;
            for (size_t k = next_op; k < o1; k++) {
                const CellOp &o = plan.ops[k];
                if (o.n > 0) {
                    first_line = std::min(first_line, o.at / kFastOpLen);
                    last_line = std::max(last_line, (o.at + o.n - 1) / kFastOpLen);
                }
                if (o.ap >= 0 && o.ap != ap) {
                    ap = o.ap;
                    first_line = std::min(first_line, o.ap / kFastOpLen);
                    last_line = std::max(last_line, o.ap / kFastOpLen);
                }
            }
            body << "            {\n"
                 << "#pragma clang fp contract(off)\n"
                 << "                FastP f = fast_get(p);\n"
                 << "                FastE ef = en;\n"
                 << "                LaneMask bad = 0;\n"
                 << "                double k2 = 0, r2 = 0;\n";
            int32_t at_line = first_line - 1;
            if (!carry && last_line >= 0)
                body << "                OpVec l" << first_line << " = load_op(cell + " << first_line * kFastOpLen << ");\n";
            auto val = [&](int32_t i) {
                return "l" + std::to_string(i / kFastOpLen) + "[" + std::to_string(i % kFastOpLen) + "]";
            };
            auto reach = [&](int32_t i) {  // value i's line: wait for it, then load the next
                while (at_line < i / kFastOpLen) {
                    at_line++;
                    body << "                arrive(l" << at_line << ");\n";
                    if (!carry && at_line == last_line) continue;
                    const int32_t nx = carry ? (at_line + 1) % plan.lines : at_line + 1;
                    body << "                " << (nx == 0 ? "" : "OpVec ") << "l" << nx << " = load_op(cell + "
                         << (at_line + 1) * kFastOpLen << ");\n"
                         << "                load_fence();\n";
                }
            };
            ap = -1;
            for (size_t k = next_op; k < o1; k++) {
                const CellOp &o = plan.ops[k];
                if (o.rad.cols || o.rad.damp) {
                    write_radiation(body, o, k, reach, val);
                    continue;
                }
                const int32_t nv = o.n;
                if (o.ap >= 0 && o.ap != ap) {
                    ap = o.ap;
                    reach(o.ap);
                    body << "                k2 = " << val(o.ap) << ";\n                r2 = " << val(o.ap + 1) << ";\n";
                }
                if (nv > 0) reach(o.at);
                body << "                {\n                    const double v[6] = {";
                for (int32_t i = 0; i < 6; i++) body << (i ? ", " : "") << (i < nv ? val(o.at + i) : "0.0");
                body << "};\n                    fast_op<maps_rad(kRare)>(f, ef, " << o.code
                     << "u, v, k2, r2, L.sp, maps_rad(kRare)" << (mixed ? " || near" : "") << ", ra, bad);\n                }\n";
            }
            // the next cell's first line is loaded behind the last one, also where no value lies in that
            // (a cell of one line, padded to two)
            if (carry) reach(plan.lines * kFastOpLen - 1);
            if (open) body << "                fast_unstable(f, ef, bad);\n";
            body << "                if (!bad) {\n"
                 << "                    put(p, en, f, ef);\n"
                 << "                } else {\n"
                 << "                    if (!this_lane(bad)) put(p, en, f, ef);\n"
                 << "                    who = bad;\n"
                 << "                    " << leave(j, j1) << '\n'
                 << "                }\n"
                 << "            }\n";
            n_seg++;
        } else {
            body << "                ;\n";
            n_seg++;
        }
        next_op = o1;
        j = j1;
    }
    std::ostringstream s;
    s << "#include <stdint.h>\n"
      << bmx_jit_src_table << '\n'
      << bmx_jit_src_maps << '\n'
      << bmx_jit_src_fast << '\n'
      << bmx_jit_src_tiles << '\n'
      << "namespace bmx {\n"
      << "struct CellTurn {\n"
      << "    static constexpr int kRare = " << maps.rare << ";\n"
      << "    __device__ __forceinline__ static void put(Particle &p, FastE &en, const FastP &f, const FastE &ef)\n"
      << "    {\n"
      << "        fast_put(p, f);\n"
      << "        if constexpr (maps_rad(kRare)) {\n"
      << "            en = ef;\n"
      << "            fast_put_energy(p, ef);\n"
      << "        }\n"
      << "    }\n"
      << "    __device__ __forceinline__ static void turn(Particle &p, const LatDesc &L, int32_t t_abs)\n"
      << "    {\n"
      << "        const CP cells = (CP)L.cell;\n"
      << "        FastE en = fast_energy(p, L.sp);\n"
      << "        const RadAt ra = {(CP)L.rad, p.id, t_abs};\n"
      << "        bool near = !maps_rad(kRare) && near_zero<kRare>(p);\n"
      << "        int32_t c = 0, seg = 0, e0 = 0, e1 = " << pd.H << ";\n"
      << "        LaneMask who = ~(LaneMask)0;\n"
      << "        bool stepwise = true, done = false;\n"
      << "        for (;;) {\n"
      << "            c = __builtin_amdgcn_readfirstlane(c);\n"
      << "            seg = __builtin_amdgcn_readfirstlane(seg);\n"
      << "            e0 = __builtin_amdgcn_readfirstlane(e0);\n"
      << "            e1 = __builtin_amdgcn_readfirstlane(e1);\n"
      // elements [e0, e1) for the lanes of who
      << "            if (e0 < e1) {\n"
      << "                if (this_lane(who)) {\n"
      << "                    track_range_fast<kRare>(p, en, L, e0, e1, t_abs, stepwise);\n"
      << "                }\n";
    // (lanes lost in an element written out come here with an empty range)
    if (mixed) s << "            }\n            {\n";
    s << "                if (p.state != ST_ALIVE) break;\n"
      << "                near = !maps_rad(kRare) && near_zero<kRare>(p);\n"
      << "            }\n"
      << "            if (done) break;\n";
    // a wave with a lane near the zero orbit goes on by the tables, which have the semi-linear bend
    if (!mixed)
        s << "            if (near) {\n"
          << "                e0 = e1;\n"
          << "                e1 = L.n_ele;\n"
          << "                who = ~(LaneMask)0;\n"
          << "                stepwise = false;\n"
          << "                done = true;\n"
          << "                continue;\n"
          << "            }\n";
    s << "            stepwise = true;\n"
      << "            who = 0;\n";
    if (carry) s << "            OpVec l0 = load_op(cells + c * " << plan.lines * kFastOpLen << ");\n";
    s << "            for (; c < " << pd.N << "; ++c) {\n"
      << "                c = __builtin_amdgcn_readfirstlane(c);\n"
      << "                const CP cell = cells + c * " << plan.lines * kFastOpLen << ";\n"
      << "                const int32_t eb = " << pd.H << " + c * " << pd.P << ";\n"
      << "                const CP base = (CP)L.prm + (" << t.hdr[pd.H].off << " + c * " << pd.S << ");\n"
      << "                switch (seg) {\n"
      << body.str()
      << "                default: seg = 0;\n"
      << "                }\n"
      << "                if (who) break;\n"
      << "            }\n"
      << "            if (!who) {\n"
      << "                e0 = " << pd.H + pd.N * pd.P << ";\n"
      << "                e1 = L.n_ele;\n"
      << "                who = ~(LaneMask)0;\n"
      << "                stepwise = false;\n"
      << "                done = true;\n"
      << "            }\n"
      << "        }\n"
      << "    }\n"
      << "};\n"
      << "}  // namespace bmx\n";
    const char *args =
        "(const bmx::Group *__restrict__ g, const bmx::WaveTile *__restrict__ t, "
        "const uint32_t *__restrict__ nt, const double *__restrict__ pi, double *__restrict__ po, "
        "uint32_t ps, uint32_t *__restrict__ co, uint32_t *tc, int32_t off, int32_t K, "
        "unsigned long long *w)";
    // the stepped quadrupole and the general bend need the 2-wave budget; a lattice that is on
    // the stepped-element map sets only for its radiation kicks gets the variants asked for
    for (int w = 3; w <= 5; w++)
        s << "extern \"C\" __global__ void __launch_bounds__(bmx::kBlock) "
          << "__attribute__((amdgpu_waves_per_eu(" << (maps.q_kinds ? 2 : w) << "))) bmx_cell_tiles_" << w << args
          << "\n{\n    bmx::track_tiles<true, bmx::CellTurn>(g, t, nt, pi, po, ps, co, tc, off, K, w);\n}\n";
    return s.str();
}

std::mutex g_mutex;
std::map<std::pair<int, std::string>, std::unique_ptr<JitKernels>> g_cache;

}  // namespace

int jit_specialize(int device, const HostTable &t, const JitKernels **out,
                   std::vector<double> &stream, std::string &err)
{
    *out = nullptr;
    Period pd;
    if (!find_period(t, pd)) {
        err = "no repeated cell covering three quarters of the lattice";
        return BMX_ERR_UNSUPPORTED;
    }
    const CellPlan plan = plan_cell(t, pd);
    const CellMaps maps = cell_maps(t);
    // the cells' values in the plan's places, and a line that the last cell's loads may reach
    stream.assign((size_t)kFastOpLen * ((size_t)plan.lines * pd.N + 1), 0.0);
    for (int32_t c = 0; c < pd.N; c++)
        for (const CellOp &o : plan.ops) {
            double *to = &stream[(size_t)kFastOpLen * plan.lines * c];
            const double *r = op_record(t, pd, c, o);
            const std::vector<double> v = op_values(t, pd, c, o);
            std::copy(v.begin(), v.end(), to + o.at);
            if (o.ap >= 0) {
                to[o.ap] = r[6];
                to[o.ap + 1] = r[7];
            }
        }
    std::lock_guard<std::mutex> lock(g_mutex);
    auto &slot = g_cache[{device, signature(t, pd, plan, maps)}];
    if (slot) {
        *out = slot.get();
        return BMX_OK;
    }
    const std::string src = generate(t, pd, plan, maps);
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), "bmx_cell.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) {
        err = "hiprtcCreateProgram failed";
        return BMX_ERR_HIP;
    }
    const char *opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=fast-honor-pragmas",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult rc = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
    if (rc != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(prog, &log[0]);
        err = std::string("cell kernel compilation failed: ") + log.substr(0, 2000);
        hiprtcDestroyProgram(&prog);
        return BMX_ERR_HIP;
    }
    size_t size = 0;
    hiprtcGetCodeSize(prog, &size);
    std::vector<char> code(size);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    auto k = std::make_unique<JitKernels>();
    k->rare_q = t.rare_q;
    k->level = t.rare_q ? (t.rad ? 2 : 1) : 0;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipModuleLoadData(&k->module, code.data());
    for (int w = 3; w <= 5 && e == hipSuccess; w++) {
        const std::string name = "bmx_cell_tiles_" + std::to_string(w);
        e = hipModuleGetFunction(&k->fn[w - 3], k->module, name.c_str());
    }
    if (e != hipSuccess) {
        err = std::string("cell kernel load: ") + hipGetErrorString(e);
        return BMX_ERR_HIP;
    }
    slot = std::move(k);
    *out = slot.get();
    return BMX_OK;
}

bool jit_rare_q(const JitKernels *j) { return j && j->rare_q; }
int jit_level(const JitKernels *j) { return j ? j->level : 0; }

hipError_t jit_occupancy(const JitKernels *j, int waves, int *blocks_per_cu)
{
    const int w = waves < 3 ? 3 : (waves > 5 ? 5 : waves);
    return hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, j->fn[w - 3], kTileBlock, 0);
}

hipError_t launch_track_tiles_jit(const JitKernels *j, hipStream_t s, int grid, int waves,
                                  const Group *d_groups, const WaveTile *d_tiles,
                                  const uint32_t *d_n_tiles, const double *d_pk_in,
                                  double *d_pk_out, uint32_t stride, uint32_t *d_cnt_out,
                                  uint32_t *d_tile_ctr, int32_t chunk_off, int32_t chunk_turns,
                                  unsigned long long *d_work)
{
    if (grid <= 0) return hipSuccess;
    const int w = waves < 3 ? 3 : (waves > 5 ? 5 : waves);
    void *args[] = {&d_groups, &d_tiles,   &d_n_tiles,  &d_pk_in,     &d_pk_out, &stride,
                    &d_cnt_out, &d_tile_ctr, &chunk_off, &chunk_turns, &d_work};
    return hipModuleLaunchKernel(j->fn[w - 3], (unsigned)grid, 1, 1, kTileBlock, 1, 1, 0, s, args,
                                 nullptr);
}

}  // namespace bmx
