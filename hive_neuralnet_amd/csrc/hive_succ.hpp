// hive_succ.hpp -- successor features of a root's legal moves, one lane per
// distinct child board.
//
// successor_row (hive_phases.hpp) gives a whole 32-lane group to one child:
// it applies the move on the LDS board and rebuilds every table of the child,
// most of them with a few lanes busy.  Here the group keeps the *root's*
// board and tables in LDS and its lanes take the root's children side by
// side: a child differs from its root in at most two cells, so each lane
// reads the root's tables and patches what it reads (struct Child).  Control
// flow over the root's pieces is the same in every lane of the group.
//
// Children whose boards differ only in the type of a piece just placed (the
// slots of one placement cell) share everything but a few counters, so they
// are one *unit*: a lane works a unit out once, and the group then writes the
// rows of each unit, adding the placed type's own contributions per row.
//
// What bounds it: VALU issue for half of the time (76 instructions a row of 427 K
// mid-game rows: 127 K of a SIMD's 249 K cycles), and the passes' serial chains --
// LDS round trips, floods, moves tried one after another -- which the 2.5 waves a
// SIMD that are left on average do not cover; the longest lists end the launch.
// 426 K mid-game rows: successor_row (about 300 VALU instructions a row) 439 us,
// here 136 us as features and 111-114 us as the units' records.
#pragma once

#include "hive_phases.hpp"

namespace hw {

constexpr int kUnits = kW;       // units of one pass: one per lane of the group
constexpr int kWinRows = 2 * kW;  // rows looked at per pass: two per lane
constexpr int kNone = -1000;      // no cell

// direction bit of cell g as seen from x by g - x + 23 (47: none), and the
// ground-slide exits of a cell by its occupied-neighbour mask, whole ring on
// the grid
struct SuccTables {
    uint8_t dir[48];
    uint8_t exits[64];
};
constexpr SuccTables make_succ_tables() {
    SuccTables t{};
    t.dir[24] = 1; t.dir[1] = 2; t.dir[0] = 4; t.dir[22] = 8; t.dir[45] = 16; t.dir[46] = 32;
    for (uint32_t n = 0; n < 64; n++) {
        const uint32_t l = ((n << 1) | (n >> 5)) & 63u, r = ((n >> 1) | (n << 5)) & 63u;
        t.exits[n] = (uint8_t)(~n & 63u & (l ^ r));
    }
    return t;
}
static __constant__ SuccTables kSuccTables = make_succ_tables();

// What the rows of one unit share: the child's 122 features, packed.  Classes
// are k = (type - 1) * 2 + colour; "2-bit" fields hold class k's small number
// at bits 2k, 2k + 1 (a board covered here has at most 3 pieces of a class).
// A placement's record leaves out what depends on the placed type, which each
// of its rows adds (row_unit).
struct alignas(4) Unit {
    uint32_t cnt;      // 2-bit: top pieces
    uint32_t hand;     // 2-bit: pieces in hand
    uint32_t near;     // 2-bit: top pieces next to the opposing queen
    uint32_t pin;      // 2-bit: pinned top pieces
    uint32_t dn;       // 2-bit: pieces with an opposing queen on the board
    uint32_t bn;       // can-move bit per class | placement cells << 16
    uint32_t dsum[4];  // byte k: distances of class k's pieces to the opposing queen, added up
    uint32_t m;        // features 96 + i that are 0 or 1 at bit i: lone piece [2], covered queen [2], (4-7), capable
                       // [2], (10-13), queens' rings of 1..6 [2][6]; the other bits are flags (kU*)
    uint32_t lift;     // throwable pieces [2], threatened pieces [2] (a byte each)
    uint32_t t;        // turn | distance of the placed piece to the opposing queen << 16
};
enum : uint32_t {
    kUNext = 1u << 4,      // black moves next
    kUPlace = 1u << 5,     // a placement: its rows add their type's share
    kUNear = 1u << 6,      // ... the placed piece is next to the opposing queen
    kUDist = 1u << 7,      // ... and has an opposing queen on the board
    kUGeneral = 1u << 10,  // not a child this program covers: successor_row's work
};

// Facts of the root (in LDS: every lane reads them, few at a time).
struct SuccRoot {
    uint32_t all;      // vertices (ranks below n)
    uint32_t one;      // one piece high
    uint32_t tall;     // stacked
    uint32_t cov[2];   // stacks that cover a queen, by its colour
    uint32_t visit;    // vertices that can matter to the next player's moves or to pillbug abilities: its own tops,
                       // stacks (what a leaving top reveals), mosquitoes and pillbugs
    uint32_t cnt, hand, dn;  // 2-bit fields of the root (Unit)
    int mosq;          // cell of the next player's mosquito on top of a single-piece cell, else kNone
    int pill;          // cell of its pillbug on top, else kNone
    int rlo, rhi;      // grid rows of the hive (empty board: the first move's row)
    uint8_t covered;   // a board this program covers
    uint8_t border;    // an occupied cell on the grid's border
    uint8_t place_any;  // the next player may place a piece
    uint8_t queen_down;  // the next player's queen is on the board
};

// A lane group's LDS: the root's board (its sm array holds the ring bytes:
// occupied on-grid neighbours in bits 0-5, bit 6 on border cells; the units
// lie over u1, u2 and the bytes after them) and the root's tables.
struct SuccBoard {
    Pos P;
    uint8_t units_end[288];
    uint32_t adj[32];             // occupied-cell graph by rank
    uint32_t info[32];            // vertex: cell | top piece << 16 | height << 24
    uint32_t row_w[25], row_b[25];  // white / black top cells of grid row r at index r + 1
    uint32_t c1[kArtN], c2[kArtN];  // components left by taking vertex v out (units_pins)
    uint32_t vert[16];            // vertices by class of their top piece
    uint32_t dist[16];            // by class: distance sum to the opposing queen | top pieces << 16 | covered pieces << 24
    uint32_t dsum[4];             // the sums as Unit::dsum
    SuccRoot R;
    uint16_t rtp[kWinRows];       // type and piece of each row of the window
    uint8_t runit[kWinRows];      // its unit
    uint16_t utp[kUnits], ufrom[kUnits], uto[kUnits];
    uint8_t urow[kUnits];         // first row of each unit
    __device__ __forceinline__ Unit* units() { return reinterpret_cast<Unit*>(&P.u1); }
};
static_assert(offsetof(Pos, u2) == offsetof(Pos, u1) + sizeof(((Pos*)nullptr)->u1) &&
                  sizeof(Unit) * kUnits <= sizeof(Pos) - offsetof(Pos, u1) + sizeof(((SuccBoard*)nullptr)->units_end) &&
                  offsetof(SuccBoard, units_end) == sizeof(Pos) && offsetof(Pos, u1) % 4 == 0,
              "the units lie over u1, u2 and units_end");

// ---------------------------------------------------------------- root
// Ring bytes (P.sm) for the rows of the hive grown by two rows each way
// (everything a child's piece can reach in a move, and that cell's
// neighbours), the occupied-cell graph.
HW_INL void build_rings(SuccBoard& G, int lane, int rlo, int rhi) {
    Pos& P = G.P;
    const int l = gl(lane);
    if (l < P.n_occ) {
        const int c = P.occ_cells[l];
        const uint64_t win = bit_window(P.occ, c - 23);
        const uint32_t nm = ring_bits(win) & grid6(c);
        const uint32_t lo = (uint32_t)win, hi = (uint32_t)(win >> 24);
        const int up = __popc(lo & 0x7FFFFEu), dn = __popc(hi & 0x1FFFFFu);
        const int rk[6] = {l + 1, l - up, l - up - (int)(lo & 1u), l - 1, l + 1 + dn, l + 1 + dn + (int)((hi >> 21) & 1u)};
        uint32_t a = 0;
#pragma unroll
        for (int d = 0; d < 6; d++)
            if (((nm >> d) & 1u) && rk[d] < kArtN) a |= 1u << rk[d];
        G.adj[l] = a;
    } else {
        G.adj[l] = 0;
    }
    const int a = rlo > 2 ? rlo - 2 : 0, b = rhi < kGrid - 3 ? rhi + 2 : kGrid - 1;
    const int g0 = (kGrid * a) >> 2, g1 = (kGrid * b + kGrid - 1) >> 2;
    uint32_t* out = reinterpret_cast<uint32_t*>(P.sm);
    for (int g = g0 + l; g <= g1; g += kW) {
        const uint64_t win = bit_window(P.occ, 4 * g - 23);
        const uint32_t wl = (uint32_t)win, wh = (uint32_t)(win >> 32);
        const uint32_t n = spread4((wl >> 24) & 15u) | (spread4((wl >> 1) & 15u) << 1) | (spread4(wl & 15u) << 2) |
                           (spread4((wl >> 22) & 15u) << 3) | (spread4((wh >> 13) & 15u) << 4) |
                           (spread4((wh >> 14) & 15u) << 5);
        const uint32_t gm = kGridBytes.w[g];
        // bit 6 of a byte whose ring is not all on the grid: 63 + 1 reaches it exactly for whole rings
        const uint32_t edge = ~((gm + 0x01010101u)) & 0x40404040u;
        out[g] = (n & gm) | edge;
    }
}

// The root's tables from a loaded board, in three steps with a barrier
// between them (`go`: this group has a new root; the other group of the wave
// only keeps the barriers).
HW_INL void succ_root(SuccBoard& G, const uint8_t* __restrict__ S, int lane, bool go) {
    Pos& P = G.P;
    const int l = gl(lane);
    if (go) {
        build_occ_list(P, lane);
        if (l < 16) G.vert[l] = G.dist[l] = 0;
    }
    __syncthreads();
    if (go) {
        SuccRoot R;
        const int me = P.turn & 1, next = me ^ 1, n = P.n_occ;
        const uint32_t rw = l < kGrid ? word_field(P.wt, kGrid * l) & 0x7FFFFFu : 0u;
        const uint32_t rb = l < kGrid ? word_field(P.bt, kGrid * l) & 0x7FFFFFu : 0u;
        if (l < kGrid + 1) {
            G.row_w[l + 1] = rw;
            G.row_b[l + 1] = rb;
        } else if (l == kGrid + 1) {
            G.row_w[0] = G.row_b[0] = 0;
        }
        const uint32_t rows = grp_ballot(l < kGrid && (word_field(P.occ, kGrid * l) & 0x7FFFFFu) != 0, lane);
        R.rlo = rows ? __ffs(rows) - 1 : kGrid / 2;
        R.rhi = rows ? 31 - __clz(rows) : kGrid / 2;
        build_rings(G, lane, R.rlo, R.rhi);
        bool bad = false, single = false, mp = false, mine = false, own = false, bug = false;
        uint32_t cover = 0;
        int c = 0;
        if (l < n) {
            c = P.occ_cells[l];
            const int h = P.hgt(c), tb = P.tp(c), pt = tb & 15, col = (tb >> 4) & 1;
            bad = pt < PT_Q || pt > PT_P || h < 1 || h > 5;
            single = h == 1;
            mp = pt == PT_M || pt == PT_P;
            own = col == next;
            mine = pt == PT_M && own && single;
            bug = pt == PT_P && own;
            if (!bad) {
                const int cls = (pt - 1) * 2 + col, q = P.queen[col ^ 1];
                atomicOr(&G.vert[cls], 1u << l);
                G.info[l] = (uint32_t)c | ((uint32_t)tb << 16) | ((uint32_t)h << 24);
                if (q < kCells) atomicAdd((int*)&G.dist[cls], hex_distance(c, q) | (1 << 16));
                for (int lv = 0; lv < h - 1; lv++) {  // under the top
                    const int b = S[lv * kCells + c], t = b & 15;
                    if (t == PT_Q && pt != PT_Q) cover |= 1u << ((b >> 4) & 1);
                    if (t < PT_Q || t > PT_P) bad = true;
                    else atomicAdd((int*)&G.dist[(t - 1) * 2 + ((b >> 4) & 1)], 1 << 24);
                }
            }
        }
        R.all = n < 32 ? (1u << n) - 1u : ~0u;
        R.one = grp_ballot(single, lane);
        R.tall = R.all & ~R.one;
        R.cov[0] = grp_ballot(cover & 1u, lane);
        R.cov[1] = grp_ballot((cover >> 1) & 1u, lane);
        R.visit = grp_ballot(mp || own, lane) | R.tall;
        const uint32_t mm = grp_ballot(mine, lane), pb = grp_ballot(bug, lane);
        R.mosq = mm ? P.occ_cells[__ffs(mm) - 1] : kNone;
        R.pill = pb ? P.occ_cells[__ffs(pb) - 1] : kNone;
        R.border = grp_ballot(l < 18 && (P.occ[l + 1] & kEdgeMask.m[l]) != 0u, lane) != 0;
        // a recorded queen's cell is in the rows whose ring bytes are built: the hive's and two more each way
        auto queen_ok = [&](int q) {
            const int r = row_of(q);
            return q == 0xFFFF || (q < kCells && r >= R.rlo - 2 && r <= R.rhi + 2);
        };
        const int turn = (P.turn + 1) & 0xFFFF;
        bad |= n > kArtN || P.result != 0 || turn == 0 || !queen_ok(P.queen[0]) || !queen_ok(P.queen[1]);
        R.queen_down = (P.qplaced >> next) & 1;
        const uint32_t held = hand_mask(P, next);
        const bool queen_now = (turn >> 1) == 3 && !R.queen_down;
        R.place_any = ((queen_now ? (held & 1u) : held) & ~((turn >> 1) == 0 ? 1u : 0u)) != 0;
        // the classes' small numbers: a class with more pieces than a set has is no game's board
        uint32_t cnt = 0, hand = 0, dn = 0, sum = 0;
        hw_group_lockstep();
        if (l < 16) {
            constexpr uint32_t kSet = 1u | (3u << 2) | (3u << 4) | (2u << 6) | (2u << 8) | (1u << 10) | (1u << 12) | (1u << 14);
            const uint32_t most = (kSet >> (2 * (l >> 1))) & 3u, h = P.hand[l & 1][l >> 1], k = __popc(G.vert[l]);
            bad |= k + h + (G.dist[l] >> 24) > most;
            cnt = (k & 3u) << (2 * l);
            hand = (h & 3u) << (2 * l);
            dn = ((G.dist[l] >> 16) & 3u) << (2 * l);
            sum = (G.dist[l] & 255u) << (8 * (l & 3));
        }
        R.covered = grp_ballot(bad, lane) == 0;
        R.cnt = grp_or(cnt);
        R.hand = grp_or(hand);
        R.dn = grp_or(dn);
        sum |= __shfl_xor(sum, 1, 64);
        sum |= __shfl_xor(sum, 2, 64);
        if (l < 16 && (l & 3) == 0) G.dsum[l >> 2] = sum;
        if (l == 0) G.R = R;
    }
    __syncthreads();
}

// ---------------------------------------------------------------- child
// A child of the group's root as one lane sees it: the root's tables, patched
// at the cell a piece left (from; vac when that emptied it) and the cell it
// reached (to; fil when that was empty).
struct Child {
    const Pos& P;
    const SuccTables& K;
    int from, to, vac, fil;
    int top_to, top_from;  // top pieces there now
    int stun;
    uint32_t pin;  // pinned root vertices
    __device__ __forceinline__ uint32_t dir(int g, int x) const {  // direction bit of g from x (off-grid pairs included)
        const uint32_t w = (uint32_t)(g - x + 23);
        return K.dir[w < 47u ? w : 47u];
    }
    __device__ __forceinline__ uint32_t grid(int x) const { return (P.sm[x] & 64u) ? grid6(x) : 63u; }
    __device__ __forceinline__ uint32_t ring(int x, uint32_t& gm) const {  // occupied on-grid neighbours of x
        const uint32_t s = P.sm[x];
        gm = 63u;
        if (s & 64u) gm = grid6(x);
        return (s & 63u & ~dir(vac, x)) | (dir(fil, x) & gm);
    }
    __device__ __forceinline__ uint32_t nb(int x) const {
        uint32_t gm;
        return ring(x, gm);
    }
    __device__ __forceinline__ uint32_t exits(int x) const {  // ground slides out of x
        uint32_t gm;
        const uint32_t n = ring(x, gm);
        return K.exits[n] & gm;
    }
    __device__ __forceinline__ uint32_t exits_without(int x, int c) const {  // ... with the piece at c lifted
        uint32_t gm;
        const uint32_t n = ring(x, gm) & ~dir(c, x);
        return K.exits[n] & gm;
    }
    __device__ __forceinline__ int hgt(int x) const {
        return P.hgt(x) - (x == from ? 1 : 0) + (x == to ? 1 : 0);
    }
    __device__ __forceinline__ int tp(int x) const { return x == to ? top_to : x == from ? top_from : P.tp(x); }
    __device__ __forceinline__ bool occ(int x) const { return (pb_get(P.occ, x) && x != vac) || x == fil; }
    __device__ __forceinline__ bool pinned(int x) const {  // x occupied
        return x != fil && ((pin >> (occ_rank(P, x) & 31)) & 1u);
    }
    __device__ __forceinline__ uint32_t heights(int x, uint32_t gm) const {  // of the six neighbours, 4 bits each
        uint32_t r = 0;
#pragma unroll
        for (int d = 0; d < 6; d++)
            if ((gm >> d) & 1u) r |= (uint32_t)(hgt(step(x, d)) & 15) << (4 * d);
        return r;
    }
};

// Existence of a move, by piece type: has_*_move (move_gen.cuh:214-1049) on the child.
HW_INL bool child_hops(const Child& V, int c) {
    uint32_t m = V.nb(c);
    const int r0 = row_of(c), q0 = c - r0 * kGrid;
    while (m) {
        const int d = __ffs(m) - 1;
        m &= m - 1;
        const int dc = (int)dir_byte(kOfsHi, kOfsLo, d) - 23;
        const int dr = (int)((kDRow >> (4 * d)) & 15u) - 1, dq = (int)((kDCol >> (4 * d)) & 15u) - 1;
        int p = c + dc, r = r0 + dr, q = q0 + dq;
        bool in = true;
        while (in && V.occ(p)) {
            r += dr;
            q += dq;
            in = (unsigned)r < (unsigned)kGrid && (unsigned)q < (unsigned)kGrid;
            p += dc;
        }
        if (in) return true;
    }
    return false;
}

HW_INL bool child_spider(const Child& V, int c) {
    uint32_t m1 = V.exits(c);
    while (m1) {  // steps back are the exit opposite the arrival: masked out
        const int d1 = __ffs(m1) - 1;
        m1 &= m1 - 1;
        const int p1 = c - 23 + (int)dir_byte(kOfsHi, kOfsLo, d1);
        uint32_t m2 = V.exits_without(p1, c) & ~dir_byte(kOppHi, kOppLo, d1);
        while (m2) {
            const int d2 = __ffs(m2) - 1;
            m2 &= m2 - 1;
            const int p2 = p1 - 23 + (int)dir_byte(kOfsHi, kOfsLo, d2);
            uint32_t m3 = V.exits_without(p2, c) & ~dir_byte(kOppHi, kOppLo, d2);
            m3 &= ~V.dir(c, p2);  // p3 == c
            if (m3) return true;
        }
    }
    return false;
}

HW_INL bool child_beetle(const Child& V, int c) {
    const uint32_t gm = V.grid(c), nh = V.heights(c, gm), sm = V.exits(c);
    const int below = V.hgt(c) - 1;
    for (int d = 0; d < 6; d++) {
        if (!((gm >> d) & 1u)) continue;
        const int mh = max(hof(nh, d), below);
        if (mh > 0 ? !gate_high(nh, d, mh) : (sm >> d) & 1u) return true;
    }
    return false;
}

HW_INL bool child_ladybug(const Child& V, int c) {
    const uint32_t nh0 = V.heights(c, V.grid(c));
    const int hc = V.hgt(c);
    uint32_t m1 = V.nb(c);
    while (m1) {
        const int d1 = __ffs(m1) - 1;
        m1 &= m1 - 1;
        const int p1 = step(c, d1);
        if (gate_high(nh0, d1, max(hc - 1, hof(nh0, d1)))) continue;
        const uint32_t nh1 = V.heights(p1, V.grid(p1));
        const int hp1 = V.hgt(p1);
        uint32_t m2 = V.nb(p1);
        while (m2) {
            const int d2 = __ffs(m2) - 1;
            m2 &= m2 - 1;
            const int p2 = step(p1, d2);
            if (p2 == c) continue;
            if (gate_high(nh1, d2, max(hp1, hof(nh1, d2)))) continue;
            const uint32_t g2 = V.grid(p2), nh2 = V.heights(p2, g2);
            uint32_t m3 = g2 & ~V.nb(p2);
            const int mh3 = V.hgt(p2);
            while (m3) {
                const int d3 = __ffs(m3) - 1;
                m3 &= m3 - 1;
                const int p3 = step(p2, d3);
                if (p3 == c || p3 == p1) continue;
                if (!gate_high(nh2, d3, mh3)) return true;
            }
        }
    }
    return false;
}

// piece_has_move (hive_phases.hpp), with its climb / jump shortcuts.  The
// abilities to try are a set of types -- the piece's own, or a ground
// mosquito's neighbours' -- so that each generator appears once in the code.
HW_INL bool child_moves(const Child& V, int c, int t, bool climb, bool jump) {
    uint32_t has = 1u << t;
    if (t == PT_M) {
        has = 0;
        if (V.hgt(c) > 1) {
            has = 1u << PT_B;
        } else {
            uint32_t om = V.nb(c);
            while (om) {
                const int d = __ffs(om) - 1;
                om &= om - 1;
                has |= 1u << (V.tp(step(c, d)) & 15);
            }
        }
    }
    if ((has & ((1u << PT_Q) | (1u << PT_P) | (1u << PT_A))) && V.exits(c) != 0) return true;
    if (((has >> PT_B) & 1u) && (climb || child_beetle(V, c))) return true;
    if (((has >> PT_G) & 1u) && (jump || child_hops(V, c))) return true;
    if (((has >> PT_S) & 1u) && child_spider(V, c)) return true;
    return ((has >> PT_L) & 1u) && child_ladybug(V, c);
}

HW_INL bool child_touches_pillbug(const Child& V, int c) {
    uint32_t m = V.nb(c);
    while (m) {
        const int d = __ffs(m) - 1;
        m &= m - 1;
        if ((V.tp(step(c, d)) & 15) == PT_P) return true;
    }
    return false;
}

// has_pillbug_throw_for_target (move_gen.cuh:742-769): the occupied neighbour
// of the actor a in direction dt
HW_INL bool child_throws(const Child& V, int a, int dt) {
    const int t = step(a, dt);
    if (V.hgt(t) != 1 || V.stun == t || V.pinned(t)) return false;
    const int ph = V.hgt(a), back = (dt + 3) % 6;
    const uint32_t gt = V.grid(t);
    const int lift = max(V.hgt(t) - 1, ph);
    const int cwh = ((gt >> ((back + 5) % 6)) & 1u) ? V.hgt(step(t, (back + 5) % 6)) : 0;
    const int ccwh = ((gt >> ((back + 1) % 6)) & 1u) ? V.hgt(step(t, (back + 1) % 6)) : 0;
    if (cwh > lift && ccwh > lift) return false;
    const uint32_t ga = V.grid(a), nha = V.heights(a, ga);
    uint32_t drop = ga & ~V.nb(a) & ~(1u << dt);
    while (drop) {
        const int dd = __ffs(drop) - 1;
        drop &= drop - 1;
        if (!gate_high(nha, dd, ph)) return true;
    }
    return false;
}

// Placement cells of the player to move after the lane's move: the grid rows
// around the hive, one after another, with the next and previous rows' words
// carried along.  A cell qualifies when it is empty, has a neighbour of that
// player's colour on top and none of the other's (before the second move:
// any neighbour).
HW_INL int child_places(const SuccBoard& G, int next, bool any_nb, int from, int to, bool stays,
                        int col_from, int col_to) {
    const int rf = from >= 0 ? row_of(from) : -8, rt = to >= 0 ? row_of(to) : -8;
    const uint32_t fb = from >= 0 ? 1u << (from - rf * kGrid) : 0u, tb = to >= 0 ? 1u << (to - rt * kGrid) : 0u;
    const uint32_t f_mine = stays && col_from == next ? fb : 0u, f_their = stays && col_from != next ? fb : 0u;
    const uint32_t t_mine = col_to == next ? tb : 0u, t_their = tb & ~t_mine;
    const uint32_t* mine = next ? G.row_b : G.row_w;
    const uint32_t* their = next ? G.row_w : G.row_b;
    int lo = G.R.rlo, hi = G.R.rhi;
    if (to >= 0) {
        lo = min(lo, rt);
        hi = max(hi, rt);
    }
    lo = max(lo - 1, 0);
    hi = min(hi + 1, kGrid - 1);
    auto fetch = [&](int r, uint32_t& m, uint32_t& t) {
        m = mine[r + 1];
        t = their[r + 1];
        if (r == rf) {
            m = (m & ~fb) | f_mine;
            t = (t & ~fb) | f_their;
        }
        if (r == rt) {
            m = (m & ~tb) | t_mine;
            t = (t & ~tb) | t_their;
        }
        if (any_nb) {
            m |= t;
            t = 0;
        }
    };
    uint32_t m0, t0, m1, t1, m2, t2;
    fetch(lo - 1, m0, t0);
    fetch(lo, m1, t1);
    int n = 0;
    for (int r = lo; r <= hi; r++) {
        fetch(r + 1, m2, t2);
        // neighbours of a cell (r, c): (r, c +- 1), (r - 1, c), (r - 1, c + 1), (r + 1, c), (r + 1, c - 1)
        const uint32_t nm = (m1 << 1) | (m1 >> 1) | m0 | (m0 >> 1) | m2 | (m2 << 1);
        const uint32_t nt = (t1 << 1) | (t1 >> 1) | t0 | (t0 >> 1) | t2 | (t2 << 1);
        n += __popc(nm & ~nt & ~m1 & ~t1 & 0x7FFFFFu);
        m0 = m1;
        t0 = t1;
        m1 = m2;
        t1 = t2;
    }
    return n;
}

// ---------------------------------------------------------------- units
// Bit matrix transpose over the lane group: lane i gives row i and gets column i.
HW_INL uint32_t grp_transpose(uint32_t x, int lane) {
    const int l = gl(lane);
    uint32_t m = 0x0000FFFFu;
#pragma unroll
    for (int j = 16; j > 0; j >>= 1) {
        const uint32_t y = __shfl_xor(x, j, 64);
        x = (l & j) ? (x & ~m) | ((y & ~m) >> j) : (x & m) | ((y & m) << j);
        m ^= m << (j >> 1);
    }
    return x;
}

// Articulation points of the children of a pass.  A child's graph is the
// root's without the vertex f that moved away (none for placements and for
// pieces leaving a stack) plus the vertex t it reached, joined to t's
// neighbours T.  The lanes flood the graph without f, lane v with v taken out
// as well: vertex v cuts it when the flood leaves a rest.  t heals v exactly
// when T meets every component (at most three: a cell's neighbours form at
// most three runs), and makes a vertex a cut only as its single neighbour.
// Which component of each v a vertex x lies in is kept per x (a transpose of
// the lanes' floods), so a child combines its few words of T instead of
// testing its T against every v.
//
// A vertex f with at most two neighbours, side by side, carries no path that
// avoids them (they are neighbours of each other): taking it out only takes
// it out of its component, which matters where it is a whole one, hanging on
// its single neighbour.  Those children share the root's own flood, like the
// ones that leave no vertex; each other f of the pass has one of its own
// (1.9 floods a pass on mid-game roots).  A board not in one piece without f
// is left to the general program.
HW_INL void units_pins(SuccBoard& G, const SuccTables& K, int lane, bool mine, int f, int vac, uint32_t T, bool has_t,
                       uint32_t& pin, bool& general) {
    const int l = gl(lane);
    const uint32_t all = G.R.all;
    bool plain = f >= 31;
    if (!plain && mine) {
        const uint32_t n = G.P.sm[vac] & 63u;
        plain = __popc(n) == 1 || (__popc(n) == 2 && (n & (rotl6(n))) != 0);
    }
    const int key = plain ? 31 : f;
    uint32_t left = grp_ballot(mine, lane);
    pin = 0;
    while (hw_wave_any(left != 0)) {
        const bool go = left != 0;
        const int ff = go ? grp_shfl(key, __ffs(left) - 1, lane) : 31;
        const bool same = go && mine && key == ff && ((left >> l) & 1u);
        left &= ~grp_ballot(same, lane);
        const uint32_t H = all & ~(ff < 31 ? 1u << ff : 0u);
        const uint32_t vbit = l < kArtN ? (1u << l) & H : 0u;
        const bool floods = go && (vbit || l == kW - 1);
        const uint32_t rest_of = H & ~vbit;
        auto flood = [&](uint32_t start) {
            uint32_t got = start, frontier = start;
            while (frontier) {
                const int i1 = __ffs(frontier) - 1;
                frontier &= frontier - 1;
                const int i2 = frontier ? __ffs(frontier) - 1 : i1;
                frontier &= frontier - 1;
                const uint32_t nw = (G.adj[i1] | G.adj[i2]) & rest_of & ~got;
                got |= nw;
                frontier |= nw;
            }
            return got;
        };
        uint32_t reach = 0;
        if (floods) reach = flood(rest_of & (0u - rest_of));
        const uint32_t rest = rest_of & ~reach;
        const bool whole = go && grp_shfl((int)(rest == 0), kW - 1, lane);
        const bool cut = floods && vbit && rest != 0;
        uint32_t second = rest;
        if (cut) {
            // a third component needs three separate neighbours: every other cell of the ring
            const int c = G.P.occ_cells[l];
            uint32_t n = G.P.sm[c] & 63u;
            if (ff < 31) {
                const uint32_t w = (uint32_t)((int)G.P.occ_cells[ff] - c + 23);
                n &= ~(uint32_t)K.dir[w < 47u ? w : 47u];
            }
            if (n == 21u || n == 42u) second = flood(rest & (0u - rest));
        }
        const uint32_t cuts = grp_ballot(cut, lane), three = grp_ballot(cut && second != rest, lane);
        const uint32_t in1 = grp_transpose(cut ? reach : 0u, lane), in2 = grp_transpose(cut ? second : 0u, lane);
        if (l < kArtN) {
            G.c1[l] = in1;
            G.c2[l] = in2;
        }
        __syncthreads();
        if (same) {
            const uint32_t fb = f < 31 ? 1u << f : 0u, h = all & ~fb;
            // the vertices whose first, second, third component T meets
            uint32_t m1 = 0, m2 = 0, m3 = 0;
            for (uint32_t t = has_t ? T : 0u; t; t &= t - 1) {
                const int x = __ffs(t) - 1;
                const uint32_t a = G.c1[x], b = G.c2[x];
                m1 |= a;
                m2 |= b;
                m3 |= ~(a | b) & ~(1u << x);
            }
            uint32_t open = cuts & ~(m1 & m2 & (m3 | ~three));  // not healed
            if (fb && plain) {
                const uint32_t vb = G.adj[f];  // f's neighbours: alone, f is a component of its single neighbour
                if ((vb & (vb - 1u)) == 0) {
                    const uint32_t a1 = G.c1[f], b1 = G.c2[f];
                    // which component of v was f: the others must be met, and must be two without t
                    const bool d1 = (a1 & vb) != 0, d2 = !d1 && (b1 & vb) != 0, d3 = !d1 && !d2;
                    const bool third = (three & vb) != 0;
                    const bool apart = (!d1 && !(m1 & vb)) || (!d2 && !(m2 & vb)) || (!d3 && third && !(m3 & vb));
                    const int parts = (third ? 3 : 2) - 1;
                    if ((cuts & vb) && (!apart || (!has_t && parts < 2))) open &= ~vb;
                    else if (cuts & vb) open |= vb;
                }
            }
            if (!whole || (has_t && T == 0 && h != 0)) general = true;
            pin = open;
            if (has_t && T && (T & (T - 1u)) == 0 && (h & ~T)) pin |= T;  // t hangs on one vertex
        }
        __syncthreads();
    }
}

// 2-bit field of class k
__device__ __forceinline__ uint32_t class_of(int t) { return (uint32_t)(((t & 15) - 1) * 2 + ((t >> 4) & 1)); }

// One pass over at most kUnits units (G.utp / ufrom / uto, lane u < nu): the
// unit's lane works its child out and leaves its record in LDS.
HW_INL void units_pass(SuccBoard& G, const SuccTables& K, const uint8_t* __restrict__ S, int lane, int nu) {
    const Pos& P = G.P;
    const SuccRoot& R = G.R;
    const int l = gl(lane);
    const bool mine = l < nu;
    const int me = P.turn & 1, next = me ^ 1;
    const int tp = mine ? G.utp[l] : MV_PASS, pt = tp >> 8;
    const int mv_from = mine ? G.ufrom[l] : 0, mv_to = mine ? G.uto[l] : 0;
    const int type = tp & 0xFF;
    bool general = !R.covered;
    bool place = false, moved = false;
    if (type == MV_PLACE) {
        place = true;
        if (mv_to >= kCells || pt < PT_Q || pt > PT_P) general = true;
        else if (pb_get(P.occ, mv_to) || ((R.hand >> (2u * class_of(pt | (me << 4)))) & 3u) == 0) general = true;
    } else if (type == MV_MOVE) {
        moved = true;
        if (mv_from >= kCells || mv_to >= kCells || mv_from == mv_to) general = true;
        else if (P.hgt(mv_from) < 1 || P.hgt(mv_to) >= 5) general = true;
    }
    if ((place || moved) && !general) {  // the ring bytes reach as far as moves along the hive do
        const int r = row_of(mv_to);
        if (r < R.rlo - 1 || r > R.rhi + 1) general = true;
    }
    if (general) place = moved = false;  // worked as a pass, written by the general program
    const int from = moved ? mv_from : kNone, to = (moved || place) ? mv_to : kNone;
    int top_from = 0, top_to = 0, under = 0;  // under: the piece covered at `to`
    bool stays = false;
    if (moved) {
        const int h = P.hgt(from);
        top_to = P.tp(from);
        if (h > 1) {
            stays = true;
            top_from = S[(h - 2) * kCells + from] & 31;
            const int t = top_from & 15;
            if (t < PT_Q || t > PT_P) general = true;
        }
        under = P.hgt(to) > 0 ? P.tp(to) : 0;
    } else if (place) {
        top_to = pt | (me << 4);
    }
    const int vac = moved && !stays ? from : kNone;
    const int fil = (moved || place) && under == 0 ? to : kNone;
    Child V{P, K, from, to, vac, fil, top_to, top_from, moved ? to : kNone, 0u};

    // neighbours of the reached cell and the vertex that moved away, by rank
    uint32_t T = 0;
    int f = 31;
    if (vac >= 0) f = occ_rank(P, vac) & 31;
    if (fil >= 0) {
        const uint64_t win = bit_window(P.occ, fil - 23);
        const uint32_t nm = V.nb(fil);
        const uint32_t lo = (uint32_t)win, hi = (uint32_t)(win >> 24);
        const int r = occ_rank(P, fil), up = __popc(lo & 0x7FFFFEu), dn = __popc(hi & 0x1FFFFFu);
        const int rk[6] = {r, r - up, r - up - (int)(lo & 1u), r - 1, r + dn, r + dn + (int)((hi >> 21) & 1u)};
#pragma unroll
        for (int d = 0; d < 6; d++)
            if ((nm >> d) & 1u) T |= 1u << (rk[d] & 31);
    }
    uint32_t cuts = 0;
    units_pins(G, K, lane, mine && !general, f, vac, T, fil >= 0, cuts, general);
    if (mine && general) G.units()[l].m = kUGeneral;
    if (mine && !general) {
        Unit& U = G.units()[l];
        // one piece high in the child: a revealed piece now may be, a covered one is not
        const uint32_t fbit = from >= 0 ? 1u << (occ_rank(P, from) & 31) : 0u;
        const uint32_t tbit = under ? 1u << (occ_rank(P, to) & 31) : 0u;
        const bool from_one = stays && P.hgt(from) == 2;
        V.pin = cuts & ((R.one & ~fbit & ~tbit) | (from_one ? fbit : 0u));
        {
            uint32_t pin = 0;
            const uint32_t old = V.pin & ~fbit;
#pragma unroll
            for (int k = 0; k < 16; k++) pin |= (uint32_t)__popc(G.vert[k] & old) << (2 * k);
            if (V.pin & fbit) pin += 1u << (2 * class_of(top_from));
            U.pin = pin;
        }
        // top pieces, hands, distances: the root's, with what the move changed
        const int tq = top_to & 15, tcol = (top_to >> 4) & 1;
        const bool queen = (moved || place) && tq == PT_Q;
        auto queen_cell = [&](int c) { return queen && tcol == c ? to : (int)P.queen[c]; };
        uint32_t m = next ? (uint32_t)kUNext : 0u, cnt = R.cnt, dn = R.dn, far = 0;
#pragma unroll
        for (int w = 0; w < 4; w++) U.dsum[w] = G.dsum[w];
        uint8_t* sums = reinterpret_cast<uint8_t*>(U.dsum);
        if (moved) {
            const int q = queen_cell(tcol ^ 1);
            if (q < kCells) sums[class_of(top_to)] += hex_distance(to, q) - hex_distance(from, q);
        } else if (place) {
            const int q = queen_cell(tcol ^ 1);
            m |= kUPlace;
            if (q < kCells) {
                m |= kUDist;
                far = hex_distance(to, q);
            }
        }
        if (stays) {
            const uint32_t k = class_of(top_from);
            const int q = queen_cell(((top_from >> 4) & 1) ^ 1);
            cnt += 1u << (2 * k);
            if (q < kCells) {
                dn += 1u << (2 * k);
                sums[k] += hex_distance(from, q);
            }
        }
        if (under) {
            const uint32_t k = class_of(under);
            const int q = queen_cell(((under >> 4) & 1) ^ 1);
            cnt -= 1u << (2 * k);
            if (q < kCells) {
                dn -= 1u << (2 * k);
                sums[k] -= hex_distance(to, q);
            }
        }
        U.cnt = cnt;
        U.dn = dn;
        U.hand = R.hand;
        U.t = (uint32_t)((P.turn + 1) & 0xFFFF) | (far << 16);
        // the queens' rings, the pieces next to them, the game's end
        int qplaced = P.qplaced;
        if (place && queen) qplaced |= 1 << me;
        bool ended = false;
        uint32_t near = 0;
        for (int c = 0; c < 2; c++) {
            const int q = queen_cell(c);
            if (q >= kCells) continue;
            uint32_t nm = V.nb(q);
            const int k = __popc(nm);
            if (k) m |= 1u << (13 + 6 * c + k);
            ended = ended || (((qplaced >> c) & 1) && k == 6 && V.occ(q));
            while (nm) {
                const int d = __ffs(nm) - 1;
                nm &= nm - 1;
                const int x = q - 23 + (int)dir_byte(kOfsHi, kOfsLo, d);
                const int t = V.tp(x);
                if (((t >> 4) & 1) == c) continue;
                if (place && x == to) m |= kUNear;
                else near += 1u << (2 * class_of(t));
            }
        }
        U.near = near;
        // a lone piece on the board
        const uint32_t alive = R.all & ~(vac >= 0 ? fbit : 0u);
        if (__popc(alive) + (fil >= 0 ? 1 : 0) == 1) {
            const int c = fil >= 0 ? fil : (int)P.occ_cells[__ffs(alive) - 1];
            m |= 1u << ((V.tp(c) >> 4) & 1);
        }
        // queens under a stack's top
        uint32_t cov = ((R.cov[0] & ~fbit & ~tbit) ? 1u : 0u) | ((R.cov[1] & ~fbit & ~tbit) ? 2u : 0u);
        if (stays && (top_from & 15) != PT_Q) {
            const int h = P.hgt(from) - 1;
            for (int lv = 0; lv < h - 1; lv++) {
                const int b = S[lv * kCells + from];
                if ((b & 15) == PT_Q) cov |= 1u << ((b >> 4) & 1);
            }
        }
        if (under && tq != PT_Q) {
            const int h = P.hgt(to);
            for (int lv = 0; lv < h; lv++) {
                const int b = S[lv * kCells + to];
                if ((b & 15) == PT_Q) cov |= 1u << ((b >> 4) & 1);
            }
        }
        m |= cov << 2;

        // what the next player can do: placement cells, then which classes can move
        uint32_t bucket = 0, lift = 0;
        int npos = 0;
        if (!ended && R.place_any)
            npos = child_places(G, next, P.turn == 0, from, to, stays, (top_from >> 4) & 1, tcol);
        const bool movable = !ended && R.queen_down && npos < kMaxLegal;
        const bool flat = R.tall == 0 && !under;
        const bool inner = !R.border && !(to >= 0 && grid6(to) != 63u);
        const bool pm_to = tq == PT_M || tq == PT_P;
        // the root's vertices that can matter, then the piece that moved (rank 31) when it is a mosquito or pillbug
        for (uint32_t left = R.visit | (pm_to ? 1u << 31 : 0u); left; left &= left - 1) {
            const int i = __ffs(left) - 1;
            int c = to, tb = top_to;
            if (i < 31) {
                const uint32_t v = G.info[i];
                c = (int)(v & 0xFFFFu);
                tb = (int)((v >> 16) & 31u);
                if (c == to) continue;  // covered: the piece that moved
                if (c == from) {
                    if (!stays) continue;
                    tb = top_from;
                }
            }
            const int t = tb & 15, col = (tb >> 4) & 1;
            const bool mp = t == PT_M || t == PT_P;
            if (movable && col == next) {
                const uint32_t bit = 1u << ((t - 1) * 2 + next);
                if (i < 31 && !((V.pin >> i) & 1u) && !(bucket & bit)) {
                    bool climb = false, jump = false;
                    if (t == PT_B || t == PT_G || t == PT_M) {
                        const bool touch = V.nb(c) != 0;
                        jump = inner && touch;
                        climb = V.hgt(c) == 1 && ((flat && touch) || V.exits(c) != 0);
                    }
                    if (child_moves(V, c, t, climb, jump)) bucket |= bit;
                }
                if (mp && (t == PT_P || (V.hgt(c) == 1 && child_touches_pillbug(V, c)))) {
                    uint32_t oa = V.nb(c);
                    while (oa) {
                        const int dt = __ffs(oa) - 1;
                        oa &= oa - 1;
                        if (child_throws(V, c, dt)) bucket |= 1u << class_of(V.tp(step(c, dt)));
                    }
                }
            }
            // pillbug-capable pieces and what they can lift (fnn_features.cuh:253-300)
            if (!mp || V.stun == c) continue;
            bool capable = t == PT_P;
            if (!capable && V.hgt(c) == 1) {
                uint32_t nm = V.nb(c);
                while (nm) {
                    const int d = __ffs(nm) - 1;
                    nm &= nm - 1;
                    const int x = step(c, d);
                    capable = capable || (V.stun != x && (V.tp(x) & 15) == PT_P);
                }
            }
            if (!capable) continue;
            m |= 1u << (8 + col);
            uint32_t nm = V.nb(c);
            while (nm) {
                const int d = __ffs(nm) - 1;
                nm &= nm - 1;
                const int x = step(c, d);
                if (V.stun == x) continue;
                const int xc = (V.tp(x) >> 4) & 1;
                lift += 1u << (8 * (xc == col ? col : 2 + xc));
            }
        }
        U.bn = bucket | ((uint32_t)npos << 16);
        U.m = m;
        U.lift = lift;
    }
    __syncthreads();
    // a queen that moved changes every distance to it: worked out again by the
    // whole group, lane i for vertex i, lane n for the piece that moved
    uint32_t queens = grp_ballot(mine && !general && (moved || place) && (top_to & 15) == PT_Q, lane);
    while (hw_wave_any(queens != 0)) {
        const bool go = queens != 0;
        const int u = go ? __ffs(queens) - 1 : 0;
        queens &= queens - 1;
        Unit& U = G.units()[u];
        if (go && l < 4) U.dsum[l] = 0;
        if (go && l == 4) U.dn = 0;
        __syncthreads();
        if (go && l <= P.n_occ) {
            const int utp = G.utp[u], ufrom = G.ufrom[u], uto = G.uto[u];
            const bool umoved = (utp & 0xFF) == MV_MOVE;
            const int top = umoved ? P.tp(ufrom) : (utp >> 8) | (me << 4);
            int c = uto, t = umoved ? top : 0;  // a placed piece's own share is its row's
            if (l < P.n_occ) {
                c = P.occ_cells[l];
                t = c == uto ? 0 : P.tp(c);
                if (umoved && c == ufrom) {
                    const int h = P.hgt(c);
                    t = h > 1 ? S[(h - 2) * kCells + c] & 31 : 0;
                }
            }
            if (t) {
                const int col = (t >> 4) & 1, k = (int)class_of(t);
                const int q = ((top >> 4) & 1) == (col ^ 1) ? uto : (int)P.queen[col ^ 1];
                if (q < kCells) {
                    atomicAdd((int*)&U.dsum[k >> 2], hex_distance(c, q) << (8 * (k & 3)));
                    atomicAdd((int*)&U.dn, 1 << (2 * k));
                }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- rows
// A quarter of a row's features: x[4 c + j] = feature 16 c + 4 g + j of the
// six sections c of 16 classes, x[24 + j] = feature 96 + 8 g + j (past 121:
// anything finite).  dsum: U.dsum[g].  The four quarters run the same code -- lanes that differ
// in g do not diverge -- and are what the lane groups of the network's first
// product take.  k: the class that a placement's row adds.  Divisions rounded
// as features_finish rounds them (div_exact).
HW_INL void unit_slice(const Unit& U, int g, uint32_t dsum, uint32_t k, float* x) {
    const uint32_t m = U.m;
    const bool add = (m & kUPlace) != 0;
    const uint32_t one = add ? 1u << (2 * k) : 0u;
    const uint32_t cnt = (U.cnt + one) >> (8 * g), hand = (U.hand - one) >> (8 * g);
    const uint32_t near = (U.near + ((m & kUNear) ? one : 0u)) >> (8 * g);
    const uint32_t dn = (U.dn + ((m & kUDist) ? one : 0u)) >> (8 * g);
    const uint32_t ds = dsum + ((m & kUDist) && (k >> 2) == (uint32_t)g ? (U.t >> 16) << (8 * (k & 3)) : 0u);
    const uint32_t move = U.bn >> (4 * g), pin = U.pin >> (8 * g);
    // hands by the pieces of a set: types 2 g and 2 g + 1 of 1 3 3 2 2 1 1 1
    const float pa = g == 1 ? 3.0f : g == 2 ? 2.0f : 1.0f, ra = g == 1 ? 1.f / 3.f : g == 2 ? 0.5f : 1.0f;
    const float pb = g == 0 ? 3.0f : g == 1 ? 2.0f : 1.0f, rb = g == 0 ? 1.f / 3.f : g == 1 ? 0.5f : 1.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        auto two = [&](uint32_t v) { return (float)((v >> (2 * j)) & 3u); };
        x[j] = two(cnt);
        x[4 + j] = div_exact(two(hand), j < 2 ? pa : pb, j < 2 ? ra : rb);
        x[8 + j] = two(near);
        const uint32_t n = (dn >> (2 * j)) & 3u;
        const float rn = n == 3 ? 1.f / 3.f : n == 2 ? 0.5f : 1.f;
        x[12 + j] = div_exact(div_exact((float)((ds >> (8 * j)) & 255u), (float)n, rn), 10.0f, 0.1f);
        x[16 + j] = (float)((move >> j) & 1u);
        x[20 + j] = two(pin);
    }
#pragma unroll
    for (int j = 0; j < 8; j++) x[24 + j] = (float)((m >> (8 * g + j)) & 1u);
    if (g == 0) {
        const float place = div_exact((float)(U.bn >> 16), 10.0f, 0.1f);
        const int turn = (int)(U.t & 0xFFFFu);
        const float t = div_exact((float)turn, 100.0f, 0.01f);
        x[28] = (m & kUNext) ? 0.0f : place;
        x[29] = (m & kUNext) ? place : 0.0f;
        x[30] = div_exact((float)max(200 - turn, 0), 200.0f, 0.005f);
        x[31] = t < 1.0f ? t : 1.0f;
    }
    if (g == 1) {
#pragma unroll
        for (int j = 0; j < 4; j++) x[26 + j] = (float)((U.lift >> (8 * j)) & 255u);
    }
}

// A row left to the general program carries this in its first feature (a NaN:
// no feature is one) until general_range has written it.
constexpr uint32_t kGeneralMark = 0xFFFFFFFFu;

// What a window's rows leave behind.  FeatureRows: 122 floats a row, eight
// rows at a time, four lanes each.  UnitRows: the units' records at their first
// rows, and a word per row -- rows back to the record, the class a placement's
// row adds at bit 8, kRowGeneral -- from which the network builds its operands
// (unit_slice); feat then holds the rows of the general program only.
struct FeatureRows {
    float* feat;
};
struct alignas(64) UnitRecord {
    Unit u;
    uint32_t pad[3];
};
constexpr uint32_t kRowGeneral = 1u << 31;
struct UnitRows {
    float* feat;
    UnitRecord* units;
    uint32_t* info;
};
template <class Out>
constexpr bool kToUnits = false;
template <>
inline constexpr bool kToUnits<UnitRows> = true;

// Where a row's root and slot come from: maps over the batch, or a list's rows
// in slot order (one memory round trip less).
struct MapRows {
    const int64_t *a2r, *midx;
    template <typename Ix>
    __device__ __forceinline__ void at(Ix i, int64_t& root, int64_t& slot) const {
        root = a2r[i];
        slot = midx[i];
    }
};
struct ListRows {
    int64_t root, first;  // the list's root and first row
    template <typename Ix>
    __device__ __forceinline__ void at(Ix i, int64_t& r, int64_t& slot) const {
        r = root;
        slot = (int64_t)i - first;
    }
};

// Successor features of rows [lo, hi) by one lane group, a window of at most
// kWinRows rows of one root at a time.  Both groups of the wave run the same
// number of windows.  A row whose root or slot is out of range gets zero
// features; a child outside what the units cover (a board or move no game
// reaches) is marked, and the return value says that the range has such rows.
template <typename Ix, class Rows, class Out>
HW_INL bool successor_range(SuccBoard& G, const SuccTables& K, const uint8_t* __restrict__ states,
                            const uint8_t* __restrict__ legal, const Rows& src, Ix lo, Ix hi, int64_t num_roots,
                            const uint8_t* __restrict__ zero_row, int wave_lane, const Out& dst) {
    int64_t cur = -2;  // the root whose tables are in LDS
    bool general = false;
    Ix at = lo;
    while (hw_wave_any(at < hi)) {
        const int lane = hw_opaque(wave_lane), l = gl(lane);  // lane constants stay out of the loop's registers
        // -- the window: rows of the root of row `at`, in a run
        int64_t key[2];
        uint32_t tp[2], from[2], to[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const Ix i = at + (Ix)(kW * j + l);
            const bool live = i < hi;
            int64_t r64 = -1, m64 = -1;
            if (live) src.at(i, r64, m64);
            const bool valid = (uint64_t)r64 < (uint64_t)num_roots && (uint64_t)m64 < (uint64_t)kMaxLegal;
            key[j] = live ? (valid ? r64 : -1) : -3;
            const uint8_t* m = valid ? legal + (Ix)(((Ix)r64 * (Ix)kMaxLegal + (Ix)m64) * (Ix)6) : zero_row;
            tp[j] = (uint32_t)m[0] | ((uint32_t)m[1] << 8);
            from[j] = (uint32_t)m[2] | ((uint32_t)m[3] << 8);
            to[j] = (uint32_t)m[4] | ((uint32_t)m[5] << 8);
        }
        const int64_t root = grp_shfl(key[0], 0, lane);
        const uint64_t same = (uint64_t)grp_ballot(key[0] == root, lane) |
                              ((uint64_t)grp_ballot(key[1] == root, lane) << 32);
        int rows = root == -3 ? 0 : (~same ? __ffsll((unsigned long long)~same) - 1 : 64);
        const bool work = root >= 0;
        const uint8_t* S = work ? states + (Ix)((Ix)root * (Ix)kStateBytes) : zero_row;
        const bool fresh = work && root != cur;
        if (hw_wave_any(fresh)) {
            if (fresh) load_position(G.P, S, lane);
            __syncthreads();
            succ_root(G, S, lane, fresh);
            if (fresh) cur = root;
        }
        // -- units: a row starts one unless it places another common type on
        // the cell of the row before (a queen, mosquito or pillbug changes more
        // than its class's counters, a mosquito takes its neighbours' types, and a
        // pillbug that throws the placed piece lets its class move).  A type that
        // is not in hand starts one of its own, which units_pass marks
        uint32_t head[2];
        uint32_t last_to = ~0u;
        const uint32_t mover = G.P.turn & 1;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t pt = tp[j] >> 8;
            const uint32_t w = (uint32_t)(G.R.mosq - (int)to[j] + 23), b = (uint32_t)(G.R.pill - (int)to[j] + 23);
            const bool plain = (tp[j] & 0xFFu) == MV_PLACE && to[j] < (uint32_t)kCells && pt < 8 && ((0xBCu >> pt) & 1u) &&
                               ((G.R.hand >> (2u * (((pt - 1u) * 2u + mover) & 15u))) & 3u) && !K.dir[w < 47u ? w : 47u] &&
                               !K.dir[b < 47u ? b : 47u];
            const uint32_t share = plain ? to[j] : 0xFFFFu;  // rows of one unit carry the same cell
            const uint32_t up = grp_shfl(share, (l + kW - 1) & (kW - 1), lane);
            const uint32_t prev = l == 0 ? last_to : up;
            last_to = grp_shfl(share, kW - 1, lane);
            head[j] = grp_ballot(work && kW * j + l < rows && (share == 0xFFFFu || share != prev), lane);
        }
        const uint32_t upto = (2u << l) - 1u;  // lanes up to and with this one
        int nu = __popc(head[0]) + __popc(head[1]);
        if (nu > kUnits) {  // the window ends before unit kUnits
            const bool over = ((head[1] >> l) & 1u) && __popc(head[0]) + __popc(head[1] & upto) == kUnits + 1;
            const uint32_t ob = grp_ballot(over, lane);
            rows = kW + __ffs(ob) - 1;
            head[1] &= ob - 1u;
            nu = kUnits;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int u = (j ? __popc(head[0]) : 0) + __popc(head[j] & upto) - 1;  // the row's unit
            G.rtp[kW * j + l] = (uint16_t)tp[j];
            G.runit[kW * j + l] = (uint8_t)u;
            if ((head[j] >> l) & 1u) {
                G.utp[u] = (uint16_t)tp[j];
                G.ufrom[u] = (uint16_t)from[j];
                G.uto[u] = (uint16_t)to[j];
                G.urow[u] = (uint8_t)(kW * j + l);
            }
        }
        __syncthreads();
        units_pass(G, K, S, lane, nu);

        const uint32_t me = G.P.turn & 1;
        if constexpr (kToUnits<Out>) {
            if (l < nu) {
                const Unit& U = G.units()[l];
                if (!(U.m & kUGeneral)) dst.units[at + (Ix)G.urow[l]].u = U;
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int r = kW * j + l;
                if (r >= rows) continue;
                const int u = work ? G.runit[r] : 0;
                const bool gen = !work || (G.units()[u].m & kUGeneral);
                const uint32_t k = (((uint32_t)(G.rtp[r] >> 8) - 1u) * 2u + me) & 15u;
                dst.info[at + (Ix)r] = gen ? kRowGeneral : (uint32_t)(r - G.urow[u]) | (k << 8);
                if (gen) {
                    general = true;
                    reinterpret_cast<uint32_t*>(dst.feat)[(Ix)((at + (Ix)r) * (Ix)kFeat)] = kGeneralMark;
                }
            }
        } else {
            const int g = l & 3;
            for (int r0 = 0; hw_wave_any(r0 < rows); r0 += 8) {
                const int r = r0 + (l >> 2);
                if (r >= rows) continue;
                float* out = dst.feat + (Ix)((at + (Ix)r) * (Ix)kFeat);
                float x[32];
                if (work) {
                    const Unit& U = G.units()[G.runit[r]];
                    if (U.m & kUGeneral) {
                        general = true;
                        if (g == 0) *reinterpret_cast<uint32_t*>(out) = kGeneralMark;
                        continue;
                    }
                    unit_slice(U, g, U.dsum[g], (((uint32_t)(G.rtp[r] >> 8) - 1u) * 2u + me) & 15u, x);
                } else {  // rows of no root or slot
#pragma unroll
                    for (int k = 0; k < 32; k++) x[k] = 0.0f;
                }
#pragma unroll
                for (int c = 0; c < 6; c++) {
                    *reinterpret_cast<f32x2*>(out + 16 * c + 4 * g) = f32x2{x[4 * c], x[4 * c + 1]};
                    *reinterpret_cast<f32x2*>(out + 16 * c + 4 * g + 2) = f32x2{x[4 * c + 2], x[4 * c + 3]};
                }
#pragma unroll
                for (int j = 0; j < 8; j += 2)
                    if (j < 2 || g < 3) *reinterpret_cast<f32x2*>(out + 96 + 8 * g + j) = f32x2{x[24 + j], x[25 + j]};
            }
        }
        __syncthreads();
        at += (Ix)rows;
    }
    return general;
}

// Rows [lo, hi) by successor_row, both groups of the wave together: the marked
// ones, after the wave's last successor_range (inside its loop this code took
// the kernel from 9 to 76 spilled registers), or with `every` all of them.
template <typename Ix = int64_t>
HW_INL void general_range(SuccBoard& G, const uint8_t* __restrict__ states, const uint8_t* __restrict__ legal,
                          const int64_t* __restrict__ a2r, const int64_t* __restrict__ midx, Ix lo, Ix hi,
                          int64_t num_roots, const uint8_t* __restrict__ zero_row, int lane, float* feat_out,
                          bool every = false) {
    SuccessorStream st;
    for (Ix at = lo; hw_wave_any(at < hi); at += kW) {
        const Ix i = at + (Ix)gl(lane);
        uint32_t rows = grp_ballot(
            i < hi && (every || reinterpret_cast<const uint32_t*>(feat_out)[(Ix)(i * (Ix)kFeat)] == kGeneralMark), lane);
        while (hw_wave_any(rows != 0)) {
            const Ix r = rows ? at + (Ix)(__ffs(rows) - 1) : hi;
            rows &= rows - 1u;
            successor_row<Ix>(G.P, st, states, legal, a2r, midx, r, hi, num_roots, zero_row, hw_opaque(lane), feat_out);
        }
    }
}

}  // namespace hw
