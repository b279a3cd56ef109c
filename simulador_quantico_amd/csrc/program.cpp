// Builds the interpreted kernels' programs (see program.hpp).
#include "program.hpp"

#include <algorithm>
#include <complex>
#include <cstring>
#include <type_traits>

namespace hgm {

namespace {

// Factors are multiplied together in a wider type and rounded once, to the
// amplitude type: a rotation's phases and coefficients are then as exact as
// the entries of its gate. For FP32 that is double, which leaves 2^-40 of an
// FP32 rounding (extended precision: 10 random layers at 12 qubits planned in
// 0.15 ms, in double in 0.066), for FP64 extended precision.
template <class T> using Wide = std::conditional_t<sizeof(T) == 4, double, long double>;

// Products of factors, none of which is infinite.
template <class R>
std::complex<R> mul(const std::complex<R> &a, const std::complex<R> &b) {
    return {a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real()};
}

int popc(uint64_t v) { return __builtin_popcountll(v); }

// A gate of a pass in tile coordinates of the execution shape, before it is
// placed in a stage: a pair gate or (diagonal) two conditional phases.
struct Item {
    const DevOp *d;
    int32_t kind;          // K_DENSE, K_ANTI, K_DIAG or K_DIAG_GLOBAL
    int32_t tbit;          // tile bit (K_DIAG_GLOBAL: state-index bit)
    uint32_t lmask, lval;
    uint64_t gmask, gval;
    uint32_t need, wr, rd; // tile bits to be registers, mixed, tested
};

// A physical operation on registers (coordinates of one stage).
template <class R>
struct ROp {
    bool phase;
    XKind kind;
    int bit = 0;
    uint32_t rmask = 0, rval = 0, tmask = 0, tval = 0;
    uint64_t gmask = 0, gval = 0;
    R m[8] = {0};
    int slot = 0;          // wave: phases even, gates odd
};

template <class R>
void split_cond(uint32_t mask, uint32_t val, uint32_t S, ROp<R> &o) {
    for (; mask; mask &= mask - 1) {
        const int b = __builtin_ctz(mask);
        const uint32_t v = (val >> b) & 1, below = (1u << b) - 1;
        if ((S >> b) & 1) {
            const int i = popc(S & below);
            o.rmask |= 1u << i;
            o.rval |= v << i;
        } else {
            const int j = popc(~S & below);
            o.tmask |= 1u << j;
            o.tval |= v << j;
        }
    }
}

bool is_one(double re, double im) { return re == 1.0 && im == 0.0; }

// Largest entry beside the 1 of a rotation's row: 1 for a unitary gate, up to
// the rounding of its entries.
constexpr double kMaxTurn = 1.0 + 1e-6;

// Phases x0, x1, y of modulus 1 with v[i][j] = x_i * o[i][j] * y_j (y_0 = 1)
// and every o[i][j] real; false when there are none up to the rounding of v's
// entries to double (16 units in the last place). Nonzero entries link rows to
// columns: with column 0's phase 1 the links give the others, and the fourth
// entry is the check. Every unitary matrix has them.
template <class R>
bool real_middle(const std::complex<R> v[2][2], std::complex<R> x[2], std::complex<R> *y, R o[2][2]) {
    using C = std::complex<R>;
    C row[2] = {C(1, 0), C(1, 0)}, col[2] = {C(1, 0), C(1, 0)};
    bool have_r[2] = {false, false}, have_c[2] = {true, false};
    for (int pass = 0; pass < 3; ++pass)
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 2; ++j) {
                if (have_c[j] == have_r[i] || v[i][j] == C(0, 0)) continue;
                const C u = v[i][j] / std::sqrt(std::norm(v[i][j]));
                if (have_c[j]) { row[i] = mul(u, std::conj(col[j])); have_r[i] = true; }
                else { col[j] = mul(u, std::conj(row[i])); have_c[j] = true; }
            }
    const C closing = mul(v[1][1], std::conj(mul(row[1], col[1])));
    if (std::abs(closing.imag()) > R(16 * 0x1p-52) * std::sqrt(std::norm(closing))) return false;
    if (v[0][0] != C(0, 0) && v[0][1] != C(0, 0) && v[1][0] != C(0, 0) && v[1][1] != C(0, 0)) {
        // what the fourth phase misses by is the entries' own rounding: a quarter to each
        const R miss = closing.imag() / closing.real();   // below 2^-47: e^(i miss) = 1 + i miss
        if (miss != 0) {
            row[0] = mul(row[0], C(1, -miss / 4));
            row[1] = mul(row[1], C(1, miss / 4));
            col[1] = mul(col[1], C(1, miss / 2));
        }
    }
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) o[i][j] = mul(v[i][j], std::conj(mul(row[i], col[j]))).real();
    x[0] = row[0];
    x[1] = row[1];
    *y = col[1];
    return true;
}

// U = e0 * diag(1, e1) * M * diag(1, y) with M = [[1, t0], [t1, 1]] and, where
// the off-diagonal entries are the larger, the rows of U exchanged.
template <class R>
struct Rotation {
    bool ok = false, exchanged = false;
    R t0 = 0, t1 = 0;
    std::complex<R> e0, e1, y;
};

template <class R>
Rotation<R> split_rotation(const double m[8]) {
    using C = std::complex<R>;
    Rotation<R> t;
    const C v[2][2] = {{C(m[0], m[1]), C(m[2], m[3])}, {C(m[4], m[5]), C(m[6], m[7])}};
    C x[2];
    R w[2][2];
    if (!real_middle(v, x, &t.y, w)) return t;
    const int ex = std::abs(w[0][0]) < std::abs(w[0][1]) ? 1 : 0;
    const R d0 = w[ex][0], d1 = w[1 - ex][1];   // of the new rows 0 and 1
    if (d0 == 0 || d1 == 0) return t;
    t.t0 = w[ex][1] / d0;
    t.t1 = w[1 - ex][0] / d1;
    if (!(std::abs(t.t0) <= kMaxTurn && std::abs(t.t1) <= kMaxTurn)) return t;
    t.exchanged = ex != 0;
    t.e0 = x[ex] * d0;
    t.e1 = mul(x[1 - ex], std::conj(x[ex])) * (d1 / (d0 * std::norm(x[ex])));
    t.ok = true;
    return t;
}

// The rotations of the gates seen last: circuits repeat their gates, and a
// split takes longer than the rest of a gate's record.
template <class R>
struct RotationMemo {
    static constexpr int kEntries = 16;
    struct Entry {
        double m[8];
        Rotation<R> t;
        bool used = false;
    } entry[kEntries];

    const Rotation<R> &of(const double m[8]) {
        uint64_t h = 0;
        for (int i = 0; i < 8; ++i) {
            uint64_t b;
            std::memcpy(&b, &m[i], 8);
            h = (h ^ b) * 0x9e3779b97f4a7c15ull;
        }
        Entry &e = entry[h >> 60];
        if (!e.used || std::memcmp(e.m, m, sizeof e.m)) {
            std::memcpy(e.m, m, sizeof e.m);
            e.t = split_rotation<R>(m);
            e.used = true;
        }
        return e.t;
    }
};

// Emits one item as register operations. `flip` holds the tile bits whose two
// values are exchanged in the registers (physical = logical ^ flip): an
// uncontrolled X, anti-diagonal gate or row-exchanged gate toggles its bit
// instead of moving amplitudes. `scale` is a factor of the whole state that is
// still to be applied. `split` turns unconditioned gates into rotations between
// phases, FP32 only: its phases are rounded once more per gate. In FP32 the
// error against 64 bits is 0.2 to 1.03 times that of whole gates (0.81 at 10
// random layers, 14 qubits, default tuning); in FP64 it would be up to 1.7 times
// (8.7e-16 -> 1.5e-15 there), for 1.37x the speed at 26 qubits (6.6 -> 4.8 ms).
// `compact` (build_exec_program) makes at most one record per gate or phase.
template <class R>
void emit(const Item &it, uint32_t S, bool f32, bool compact, uint32_t &flip, std::complex<R> &scale, RotationMemo<R> &memo,
          std::vector<ROp<R>> &out) {
    using C = std::complex<R>;
    const DevOp &d = *it.d;
    const uint32_t lval = it.lval ^ (flip & it.lmask);
    auto phase = [&](C f, uint32_t lm, uint32_t lv, uint64_t gm, uint64_t gv) {
        if (f == C(1, 0)) return;
        ROp<R> o;
        o.phase = true;
        o.kind = X_PHASE;
        split_cond(lm, lv, S, o);
        o.gmask = gm;
        o.gval = gv;
        o.m[0] = f.real();
        o.m[1] = f.imag();
        out.push_back(o);
    };
    if (it.kind == K_DIAG_GLOBAL) {
        for (int v = 0; v < 2; ++v)
            phase(C(d.m[6 * v], d.m[6 * v + 1]), it.lmask, lval, it.gmask | (uint64_t(1) << it.tbit),
                  it.gval | (uint64_t(v) << it.tbit));
        return;
    }
    const uint32_t tb = 1u << it.tbit, f = (flip >> it.tbit) & 1u;
    if (it.kind == K_DIAG) {
        for (uint32_t v = 0; v < 2; ++v)
            phase(C(d.m[6 * v], d.m[6 * v + 1]), it.lmask | tb, lval | ((v ^ f) << it.tbit), it.gmask, it.gval);
        return;
    }
    double m[8];   // row-major on the physical pair
    for (int row = 0; row < 2; ++row)
        for (int col = 0; col < 2; ++col)
            for (int c = 0; c < 2; ++c) m[4 * row + 2 * col + c] = d.m[4 * (row ^ (int)f) + 2 * (col ^ (int)f) + c];
    const bool free_gate = !it.lmask && !it.gmask;
    const bool split = f32 && !compact;
    const bool unit_anti = it.kind == K_ANTI && is_one(m[2], m[3]) && is_one(m[4], m[5]);
    if (it.kind == K_ANTI && free_gate && (unit_anti || !compact)) {   // values exchanged, then a phase on each
        flip ^= tb;
        phase(C(m[4], m[5]), tb, 0, 0, 0);
        phase(C(m[2], m[3]), tb, tb, 0, 0);
        return;
    }
    ROp<R> o;
    o.phase = false;
    o.bit = popc(S & (tb - 1));
    if (free_gate && split) {
        const Rotation<R> &t = memo.of(m);
        if (t.ok) {
            phase(t.y, tb, tb, 0, 0);
            if (t.exchanged) flip ^= tb;
            o.kind = X_ROT;
            o.m[0] = t.t0;
            o.m[2] = t.t1;
            out.push_back(o);
            scale = mul(scale, t.e0);
            phase(t.e1, tb, tb, 0, 0);
            return;
        }
    }
    // Rows that each hold an exact 1 (HGM_PLAN_PIVOT), in different columns: half
    // the multiply-adds, and no rounding that the whole gate does not have. 8
    // random layers at 26 qubits, complex128: 6.6 -> 5.5 ms; Grover at 22: 1.36 ->
    // 1.19. A record kind of its own beside the real rotation made the kernels
    // larger: 6 layers at 12 qubits, which run neither, 59 -> 62 us.
    if (free_gate && !f32) {
        const int ex = is_one(m[0], m[1]) && is_one(m[6], m[7]) ? 0 : is_one(m[2], m[3]) && is_one(m[4], m[5]) ? 1 : -1;
        if (ex >= 0 && it.kind != K_ANTI) {
            // rows exchanged (ex): the new row 0 is row 1, the new row 1 is row 0
            const double *t0 = m + (ex ? 6 : 2), *t1 = m + (ex ? 0 : 4);
            o.kind = X_ROT;
            std::copy(t0, t0 + 2, o.m);
            std::copy(t1, t1 + 2, o.m + 2);
            if (ex) flip ^= tb;
            out.push_back(o);
            return;
        }
    }
    split_cond(it.lmask, lval, S, o);
    o.gmask = it.gmask;
    o.gval = it.gval;
    std::copy(m, m + 8, o.m);
    const bool real = m[1] == 0 && m[3] == 0 && m[5] == 0 && m[7] == 0;
    if (o.rmask) o.kind = real ? X_REAL_MASK : X_DENSE_MASK;
    else if (unit_anti) o.kind = X_SWAP;
    else if (o.tmask) o.kind = real ? X_REAL_LANE : X_DENSE_LANE;
    else o.kind = real ? X_DENSE_REAL : X_DENSE;
    out.push_back(o);
}

// Stable insertion sort: the lists are short (kChunk) and nearly in order.
template <class I, class F>
void sort_stable(I b, I e, F less) {
    for (I i = b; i != e; ++i)
        for (I j = i; j != b && less(*j, *(j - 1)); --j) std::swap(*j, *(j - 1));
}

// Orders a stage's operations into waves (phases as early as they commute,
// then gates), keeping the order of every pair that does not commute: gates
// on a register bit conflict with gates on it and with whatever tests it.
template <class R>
void into_waves(std::vector<ROp<R>> &ops, std::vector<const ROp<R> *> &order) {
    int gate[8] = {0}, test[8] = {0};
    order.clear();
    for (ROp<R> &o : ops) {
        int s = 0;
        for (uint32_t m = o.rmask; m; m &= m - 1) s = std::max(s, gate[__builtin_ctz(m)]);
        if (!o.phase) s = std::max({s, gate[o.bit], test[o.bit]});
        if ((s & 1) == (o.phase ? 1 : 0)) ++s;
        o.slot = s;
        for (uint32_t m = o.rmask; m; m &= m - 1) test[__builtin_ctz(m)] = std::max(test[__builtin_ctz(m)], s);
        if (!o.phase) gate[o.bit] = std::max(gate[o.bit], s);
        order.push_back(&o);
    }
    sort_stable(order.begin(), order.end(), [](const ROp<R> *a, const ROp<R> *b) { return a->slot < b->slot; });
}

template <class T>
XOp<T> record(const ROp<Wide<T>> &o, uint32_t A) {
    XOp<T> x;
    std::memset(&x, 0, sizeof x);
    x.kind = (uint8_t)o.kind;
    x.bit = (uint8_t)o.bit;
    x.tmask = o.tmask;
    x.tval = o.tval;
    x.gmask = o.gmask;
    x.gval = o.gval;
    for (int i = 0; i < 8; ++i) x.m[i] = (T)o.m[i];
    if (o.phase) {
        const double g[2] = {(double)o.m[0], (double)o.m[1]};
        std::memcpy(x.m, g, sizeof g);
    }
    for (uint32_t k = 0; k < A; ++k)
        if ((o.phase || !((k >> o.bit) & 1)) && (k & o.rmask) == o.rval) x.pmask |= 1u << k;
    if (o.phase) {
        x.pat = X_PAT_MASK;
        if (popc(o.rmask) <= 2 && o.rval == o.rmask) x.pat = (uint8_t)o.rmask;
        else if (popc(o.rmask) == 1) x.pat = (uint8_t)(X_PAT_CLEAR + __builtin_ctz(o.rmask));
    }
    return x;
}

// Records of one pass, and the factors of its X_VEC records.
template <class T>
struct Records {
    using C = std::complex<Wide<T>>;
    using ROp = struct ROp<Wide<T>>;

    uint32_t A;
    bool compact;        // no factor tables
    std::vector<XOp<T>> ops;
    std::vector<T> table;
    C scale = C(1, 0);   // factor of the whole state still to be applied

    std::vector<const ROp *> order;   // scratch
    std::vector<ROp> group;
    C f[kMaxRegAmps];

    // A factor per register (f), the pending scale included.
    void vec() {
        bool real = true, one = true;
        for (uint32_t k = 0; k < A; ++k) {
            if (scale != C(1, 0)) f[k] = mul(f[k], scale);
            real = real && (T)f[k].imag() == T(0);
            one = one && f[k] == C(1, 0);
        }
        scale = C(1, 0);
        if (one) return;
        XOp<T> x;
        std::memset(&x, 0, sizeof x);
        x.kind = real ? X_VEC_REAL : X_VEC;
        x.pmask = (uint32_t)table.size();
        for (uint32_t k = 0; k < A; ++k) {
            table.push_back((T)f[k].real());
            if (!real) table.push_back((T)f[k].imag());
        }
        ops.push_back(x);
    }

    using It = typename std::vector<const ROp *>::const_iterator;

    // The phases [b, e) of a wave that test register bits only: one record when
    // a pattern of set (or one clear) register bits says it, else one factor
    // per register.
    void uniform(It b, It e) {
        if (b == e) return;
        if (compact) {
            for (; b != e; ++b) {
                XOp<T> x = record<T>(**b, A);
                x.flags = (uint8_t)(X_FIRST | X_LAST | ((*b)->m[1] == 0 ? X_REAL : 0));
                ops.push_back(x);
            }
            return;
        }
        if (e - b == 1 && scale == C(1, 0)) {
            XOp<T> x = record<T>(**b, A);
            if (x.pat != X_PAT_MASK) {
                x.flags = (uint8_t)(X_FIRST | X_LAST | ((*b)->m[1] == 0 ? X_REAL : 0));
                ops.push_back(x);
                return;
            }
        }
        std::fill(f, f + A, C(1, 0));
        for (; b != e; ++b) {
            const ROp &o = **b;
            for (uint32_t k = 0; k < A; ++k) {
                if ((k & o.rmask) != o.rval) continue;
                if (o.m[1] == 0) f[k] *= o.m[0];
                else f[k] = mul(f[k], C(o.m[0], o.m[1]));
            }
        }
        vec();
    }

    // Phases with conditions on threads or tiles, grouped by the registers they
    // act on (the caller sorted them), equal conditions multiplied together.
    void groups(It b, It e) {
        while (b != e) {
            group.clear();
            const ROp &head = **b;
            for (; b != e && (*b)->rmask == head.rmask && (*b)->rval == head.rval; ++b) {
                const ROp &o = **b;
                auto same = std::find_if(group.begin(), group.end(), [&](const ROp &g) {
                    return g.tmask == o.tmask && g.tval == o.tval && g.gmask == o.gmask && g.gval == o.gval;
                });
                if (same == group.end()) { group.push_back(o); continue; }
                const C z = mul(C(same->m[0], same->m[1]), C(o.m[0], o.m[1]));
                same->m[0] = z.real();
                same->m[1] = z.imag();
            }
            // Where no record of a group holds, its factor is 1, and an infinity times 1 + 0i is no infinity: complex
            // phases that all wait for some tile are applied one by one, each in its tiles, and real ones (whose 1
            // changes nothing) by themselves.
            const auto real = [](const ROp &g) { return g.m[1] == 0; };
            const bool everywhere = std::any_of(group.begin(), group.end(), [&](const ROp &g) { return !real(g) && !g.gmask; });
            const auto mid = everywhere ? group.end() : std::stable_partition(group.begin(), group.end(), real);
            for (auto g = group.begin(); g != group.end(); ++g) {
                XOp<T> x = record<T>(*g, A);
                const bool alone = g >= mid;
                x.flags = (uint8_t)((alone || g == group.begin() ? X_FIRST : 0) | (alone || g + 1 == mid ? X_LAST : 0) |
                                    (!alone && !everywhere ? X_REAL : 0));
                ops.push_back(x);
            }
        }
    }

    // A rotation by itself: FP32 ones are real, FP64 ones may be complex.
    XOp<T> rotation(const ROp &o) {
        XOp<T> x = record<T>(o, A);
        if (sizeof(T) == 4) x.m[1] = x.m[2];
        return x;
    }

    // A run of rotations: those on different register bits commute, and three
    // of a full set of four (two of two or three) already cost less as one
    // record than one by one.
    void rotations(It b, It e) {
        const int bits = A == 2 ? 1 : A == 4 ? 2 : A == 8 ? 3 : 4;
        while (b != e) {
            uint32_t used = 0;
            It n = b;
            for (; n != e && (*n)->bit < bits && !((used >> (*n)->bit) & 1u) && real(**n); ++n) used |= 1u << (*n)->bit;
            if (n == b) ++n;   // a fifth register bit, or complex
            if (popc(used) >= (bits + 2) / 2 && bits > 1) {
                XOp<T> x;
                std::memset(&x, 0, sizeof x);
                x.kind = X_ROTS;
                for (; b != n; ++b) {
                    x.m[2 * (*b)->bit] = (T)(*b)->m[0];
                    x.m[2 * (*b)->bit + 1] = (T)(*b)->m[2];
                }
                ops.push_back(x);
            } else {
                for (; b != n; ++b) ops.push_back(rotation(**b));
            }
        }
    }

    static bool real(const ROp &o) { return o.m[1] == 0 && o.m[3] == 0; }

    void stage(std::vector<ROp> &list) {
        into_waves(list, order);
        for (auto i = order.begin(); i != order.end();) {
            auto e = i;
            if (!(*i)->phase) {
                if ((*i)->kind != X_ROT) { ops.push_back(record<T>(**i++, A)); continue; }
                while (e != order.end() && !(*e)->phase && (*e)->kind == X_ROT) ++e;
                rotations(i, e);
                i = e;
                continue;
            }
            while (e != order.end() && (*e)->phase && (*e)->slot == (*i)->slot) ++e;
            auto uniform_op = [](const ROp *o) { return !o->tmask && !o->gmask; };
            sort_stable(i, e, [&](const ROp *a, const ROp *b) {
                if (uniform_op(a) != uniform_op(b)) return uniform_op(a);
                return a->rmask != b->rmask ? a->rmask < b->rmask : a->rval < b->rval;
            });
            auto u = i;
            while (u != e && uniform_op(*u)) ++u;
            uniform(i, u);
            groups(u, e);
            i = e;
        }
    }

    // The pending scale, when it is due: at the end of the pass, and before it
    // moves the amplitudes far from 1.
    void flush(bool end) {
        const auto s = std::norm(scale);
        if (scale == C(1, 0) || (!end && s >= 0x1p-40 && s <= 0x1p40)) return;
        std::fill(f, f + A, C(1, 0));
        vec();
    }
};

// Operations of a stage put into waves together.
constexpr size_t kChunk = 64;

// Gates of one launch of a whole-state workgroup, at most (about 10 ms).
constexpr size_t kMaxLaunchItems = size_t(1) << 15;

// Runs of an ascending bit deposit: index bit j goes to state bit pos[j].
int deposit_runs(const int *pos, int n, XRun *out, int cap) {
    int runs = 0;
    for (int j = 0; j < n;) {
        int len = 1;
        while (j + len < n && pos[j + len] == pos[j] + len && len < 32) ++len;
        if (runs < cap) out[runs] = {len >= 32 ? ~0u : (1u << len) - 1, (uint16_t)j, (uint16_t)pos[j]};
        ++runs;
        j += len;
    }
    return runs;
}

// The gates of a pass as items in tile coordinates: tile bit j is state bit
// pos[j].
void pass_items(const Plan &plan, const Pass &ps, const int *pos, int r, std::vector<Item> &items) {
    int tile_of[64];
    std::fill(tile_of, tile_of + 64, -1);
    for (int j = 0; j < r; ++j) tile_of[pos[j]] = j;
    items.reserve(items.size() + (size_t)ps.op_count);
    for (int64_t i = 0; i < ps.op_count; ++i) {
        const DevOp &d = plan.ops[ps.op_begin + i];
        Item it{&d, d.kind, d.tbit, 0, 0, 0, 0, 0, 0, 0};
        auto cond = [&](int b, uint64_t v) {   // state bit b has value v
            if (tile_of[b] >= 0) {
                it.lmask |= 1u << tile_of[b];
                it.lval |= (uint32_t)v << tile_of[b];
            } else {
                it.gmask |= uint64_t(1) << b;
                it.gval |= v << b;
            }
        };
        for (uint32_t m = d.lmask; m; m &= m - 1) cond(ps.local_pos[__builtin_ctz(m)], (d.lval >> __builtin_ctz(m)) & 1);
        for (uint64_t m = d.gmask; m; m &= m - 1) cond(__builtin_ctzll(m), (d.gval >> __builtin_ctzll(m)) & 1);
        const int target = d.kind == K_DIAG_GLOBAL ? d.tbit : ps.local_pos[d.tbit];
        if (tile_of[target] >= 0) {
            if (d.kind == K_DIAG_GLOBAL) it.kind = K_DIAG;
            it.tbit = tile_of[target];
        } else {
            it.tbit = target;
        }
        it.rd = it.lmask;
        if (it.kind == K_DENSE || it.kind == K_ANTI) it.need = it.wr = 1u << it.tbit;
        else if (it.kind == K_DIAG) {
            it.rd |= 1u << it.tbit;
            if (plan.pre_phase[ps.op_begin + i]) it.need = it.wr = 1u << it.tbit;
        }
        items.push_back(it);
    }
}

// Appends the program of one launch: `items` on tiles of 2^rx amplitudes whose
// bit j is state bit pos[j]; gates mix the first r tile bits only, and the
// first c stay on consecutive threads at the load and the store.
template <class T>
void build(Plan &plan, const std::vector<Item> &items, const int *pos, int r, int rx, int c, bool compact, RotationMemo<Wide<T>> &memo) {
    constexpr int F = sizeof(T) == 4 ? 5 : 4;
    const ExecShape &ex = plan.exec;
    const int n = plan.qubits;
    int a = 0;
    while ((1 << a) < ex.A) ++a;
    const uint32_t own = (uint32_t)((uint64_t(1) << r) - 1);
    const uint32_t forbid = (r - c >= a) ? (uint32_t)((1u << c) - 1) : 0u;
    uint64_t local = 0;
    for (int j = 0; j < rx; ++j) local |= uint64_t(1) << pos[j];
    std::vector<ROp<Wide<T>>> ops;
    ops.reserve(kChunk + 4);
    // stages: the same greedy as the pass planner, with the tile as the state and the register bits as the
    // tile; the first and last keep the coalesced bits on the threads
    std::vector<uint32_t> sets;
    std::vector<std::vector<int>> lists;
    std::vector<char> done(items.size(), 0);
    for (size_t head = 0; head < items.size();) {
        uint32_t S = 0, bw = 0, br = 0;
        int nS = 0;
        std::vector<int> list;
        for (size_t k = head; k < items.size(); ++k) {
            if (done[k]) continue;
            const Item &it = items[k];
            bool ok = !(it.wr & (bw | br)) && !(it.rd & bw);
            if (ok && (it.need & ~S)) {
                if (nS < a && !(sets.empty() && (it.need & forbid))) { S |= it.need; ++nS; }
                else ok = false;
            }
            if (ok) { list.push_back((int)k); done[k] = 1; }
            else { bw |= it.wr; br |= it.rd; if ((bw & own) == own) break; }
        }
        while (head < items.size() && done[head]) ++head;
        sets.push_back(S);
        lists.push_back(std::move(list));
    }
    if (sets.empty() || (sets.back() & forbid)) { sets.push_back(0); lists.emplace_back(); }
    for (size_t i = 0; i < sets.size(); ++i) {
        const bool edge = i == 0 || i + 1 == sets.size();
        for (int b = r - 1; b >= 0 && popc(sets[i]) < a; --b)
            if (!((sets[i] >> b) & 1) && !(edge && ((forbid >> b) & 1))) sets[i] |= 1u << b;
        for (int b = r - 1; b >= 0 && popc(sets[i]) < a; --b) sets[i] |= 1u << b;
    }
    // records
    auto map_of = [&](uint32_t S) {
        XMap m;
        std::memset(&m, 0, sizeof m);
        int i = 0;
        for (int b = 0; b < rx; ++b)
            if ((S >> b) & 1) {
                m.low[i] = (uint16_t)((1u << b) - 1);
                m.sw[i++] = (uint16_t)x_swizzle<F>(1u << b);
            }
        return m;
    };
    Records<T> recs;
    recs.A = (uint32_t)ex.A;
    recs.compact = compact;
    recs.ops.reserve(items.size() + items.size() / 2 + 16);
    uint32_t flip = 0;
    for (size_t i = 0; i < sets.size(); ++i) {
        if (i > 0) {
            XOp<T> x;
            std::memset(&x, 0, sizeof x);
            x.kind = X_REMAP;
            const XMap m = map_of(sets[i]);
            std::memcpy(x.m, &m, sizeof m);
            recs.ops.push_back(x);
        }
        ops.clear();
        for (int k : lists[i]) {
            emit(items[k], sets[i], sizeof(T) == 4, compact, flip, recs.scale, memo, ops);
            if (ops.size() >= kChunk) { recs.stage(ops); recs.flush(false); ops.clear(); }
        }
        recs.stage(ops);
        recs.flush(i + 1 == sets.size());
    }
    XPass xp;
    std::memset(&xp, 0, sizeof xp);
    xp.n_ops = (int32_t)recs.ops.size();
    xp.first = map_of(sets.front());
    auto lanes = [&](uint32_t S, uint64_t *bit, XRun *runs) {
        int p[32], np = 0, i = 0;
        for (int b = 0; b < rx; ++b) {
            if ((S >> b) & 1) bit[i++] = uint64_t(1) << pos[b];
            else p[np++] = pos[b];
        }
        return deposit_runs(p, np, runs, kXLaneRuns);
    };
    xp.n_load = lanes(sets.front(), xp.lbit, xp.load);
    xp.n_store = lanes(sets.back(), xp.sbit, xp.store);
    for (int b = 0; b < rx; ++b)
        if ((flip >> b) & 1) ((sets.back() >> b) & 1 ? xp.rflip : xp.sflip) |= uint64_t(1) << pos[b];
    int p[64], np = 0;
    for (int b = 0; b < n; ++b)
        if (!((local >> b) & 1)) p[np++] = b;
    xp.n_base = deposit_runs(p, np, xp.base, kXBaseRuns);
    // one zero record past the end (the kernel loads ahead), then the factor table
    const size_t op_bytes = (recs.ops.size() + 1) * sizeof(XOp<T>);
    const size_t table_at = (sizeof(XPass) + op_bytes + 63) / 64 * 64;
    xp.table = (int64_t)table_at;
    const size_t at = plan.xprog.size();
    plan.xprog.resize(at + (table_at + recs.table.size() * sizeof(T) + 63) / 64 * 8, 0);
    plan.xlaunch.push_back({(int64_t)(at * 8), (int32_t)((plan.xprog.size() - at) * 8), (int32_t)sets.size()});
    char *to = reinterpret_cast<char *>(&plan.xprog[at]);
    std::memcpy(to, &xp, sizeof xp);
    if (!recs.ops.empty()) std::memcpy(to + sizeof xp, recs.ops.data(), recs.ops.size() * sizeof(XOp<T>));
    if (!recs.table.empty()) std::memcpy(to + table_at, recs.table.data(), recs.table.size() * sizeof(T));
}

// The execution shape of a plan: the plan's own threads and amplitudes per
// thread, with more amplitudes per thread where the tuning asks for fewer than
// the kernel does well with, and several tiles per workgroup where a tile has
// less than a wave. 16 amplitudes per thread halve the records and the remaps
// of 8 (default tuning, random layers: 25 qubits FP32 4 / 8 / 16 amplitudes
// 3589 / 1938 / 1192 us, FP64 3910 / 2879 / 2484); up to 12 qubits a pass is
// one chain of records on few waves, and 8 make each shorter (QFT at 11
// qubits 35 / 27 / 28 us). FP64 of 13-19 qubits gains nothing either way (15
// qubits: 92 / 96 / 94).
ExecShape choose_shape(const Plan &plan, bool whole) {
    const int n = plan.qubits, r = whole ? n : plan.shape.r, c = std::min(plan.shape.c, r);
    int a = 0;
    while ((2 << a) <= 2 * plan.shape.R) ++a;
    int want = a;
    if (n <= 12) want = 3;
    else if (n >= 20 || plan.dtype == HGM_C64) want = 4;
    if (whole) a = std::max(a, n <= 12 ? std::min(3, n) : 4);
    while (a < want && a < r - c) ++a;
    ExecShape e;
    e.A = 1 << a;
    e.r = r;
    e.sync = r - a > 6;
    while (e.r - a < 6 && e.r < n) ++e.r;
    e.B = 1 << (e.r - a);
    return e;
}

// Whether one workgroup runs the whole state, all passes in one launch: their
// launches cost about 5 us each, and merged passes share remaps, while a pass
// on its own spreads its tiles over workgroups. Default tuning, FP32, passes
// on their own against one launch: Grover (8 iterations, 10-17 passes) at 9 /
// 11 / 13 qubits 108 / 115 / 182 against 47 / 71 / 112 us, random layers (3-5
// passes) 32 / 38 / 48 against 27 / 36 / 46, QFT (2-3 passes) 19 / 25 / 35
// against 17 / 24 / 38.
bool whole_state(const Plan &plan) {
    int64_t passes = 0;
    for (const Pass &ps : plan.passes) passes += ps.op_count > 0;
    return passes > 1 && (plan.qubits <= 11 || (plan.qubits <= 13 && passes >= 6));
}

}  // namespace

void build_exec_program(Plan &plan, bool pass_by_pass, bool compact) {
    const bool whole = !pass_by_pass && whole_state(plan);
    plan.exec = choose_shape(plan, whole);
    plan.xprog.clear();
    plan.xlaunch.clear();
    const int n = plan.qubits, r = whole ? n : plan.shape.r, rx = plan.exec.r;
    std::vector<Item> items;
    RotationMemo<double> memo;
    RotationMemo<long double> unused;   // FP64 programs hold whole gates
    int pos[32];
    auto launch = [&] {
        if (plan.dtype == HGM_C64) build<float>(plan, items, pos, r, rx, std::min(plan.shape.c, r), compact, memo);
        else build<double>(plan, items, pos, r, rx, std::min(plan.shape.c, r), compact, unused);
        items.clear();
    };
    for (const Pass &ps : plan.passes) {
        if (!ps.op_count) {
            if (pass_by_pass) plan.xlaunch.push_back({});   // launches are indexed by pass there
            continue;
        }
        // tile bits: the state's, or the plan's, then the lowest non-local ones
        uint64_t local = 0;
        for (int j = 0; j < r; ++j) pos[j] = whole ? j : ps.local_pos[j], local |= uint64_t(1) << pos[j];
        for (int j = r, b = 0; j < rx; ++b)
            if (!((local >> b) & 1)) { pos[j++] = b; local |= uint64_t(1) << b; }
        pass_items(plan, ps, pos, rx, items);
        if (!whole || items.size() >= kMaxLaunchItems) launch();
    }
    if (!items.empty()) launch();
}

}  // namespace hgm
