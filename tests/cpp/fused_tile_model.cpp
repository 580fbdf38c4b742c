// A CPU model of the fused kernel's tile body as it runs (qvnt_amd/csrc/
// fused.hip: fused_tile; tile.hpp), driven by the real host compiler: the
// tile read and written in the edge phases' layouts, moved through LDS from
// one phase's register layout to the next, dense phases in the matrix cores'
// layout, the permuted read-out.  It checks what the kernel relies on -- every
// amplitude read once and written once, every exchange a bijection inside
// the tile, a pass's ops one after the other, the reads one op and one phase
// ahead inside the packed program -- and that the result equals the oracle's
// plain apply.  Circuits, the ops of a phase and the comparison of programs
// are fused_model.cpp's.
#define main model_main
#include "fused_model.cpp"
#undef main

// tile.hpp: swz
static uint32_t tswz(uint32_t e) { return e ^ (e >> 4); }
static uint32_t spread(uint32_t x, const uint32_t* p) {
    for (int j = 0; j < kRegBits; ++j) {
        const uint32_t lo = x & ((1u << p[j]) - 1u);
        x = ((x ^ lo) << 1) | lo;
    }
    return x;
}
static uint32_t byte_of(uint32_t w, int k) { return (w >> (8 * k)) & 63u; }

// LDS offset of a thread's register i: base ^ bits
struct Layout {
    uint32_t base, bit[kRegBits];
    uint32_t operator()(int i) const {
        uint32_t e = base;
        for (int j = 0; j < kRegBits; ++j)
            if (i >> j & 1) e ^= bit[j];
        return e;
    }
};
static Layout layout_of(uint32_t tb, const uint32_t* p) {
    Layout l;
    l.base = tswz(tb);
    for (int j = 0; j < kRegBits; ++j) l.bit[j] = tswz(1u << p[j]);
    return l;
}
// the element behind an offset of tswz, tiles of at most 2^13
static uint32_t element(uint32_t off) {
    uint32_t e = off;
    for (int k = 0; k < 4; ++k) e = off ^ (e >> 4);
    CHECK(tswz(e) == off);
    return e;
}
static Layout dense_layout(const FPhase& ph, uint32_t tid) {
    const uint32_t hi = (tid >> 4) & 3u;
    uint32_t e = spread(tid & ~48u, ph.rpos);
    e |= ((hi & 1u) << ph.rpos[0]) | ((hi >> 1) << ph.rpos[1]);
    Layout l;
    l.base = tswz(e);
    l.bit[0] = tswz(1u << ph.rpos[2]);
    l.bit[1] = tswz(1u << ph.rpos[3]);
    l.bit[2] = tswz(spread(16u, ph.rpos));
    l.bit[3] = tswz(spread(32u, ph.rpos));
    return l;
}

// V[tid * 16 + i] from `from` to `to(tid, i)` through LDS, both one to one
template <class To>
static void exchange(std::vector<C>& V, uint32_t t, const std::vector<Layout>& from, const To& to) {
    std::vector<C> lds(1u << t);
    std::vector<char> put(1u << t, 0), got(1u << t, 0);
    for (uint32_t tid = 0; tid < from.size(); ++tid)
        for (int i = 0; i < kRegs; ++i) {
            const uint32_t o = from[tid](i);
            CHECK(o < (1u << t) && !put[o]);
            put[o] = 1;
            lds[o] = V[tid * kRegs + i];
        }
    for (uint32_t tid = 0; tid < from.size(); ++tid)
        for (int i = 0; i < kRegs; ++i) {
            const uint32_t o = to(tid, i);
            CHECK(o < (1u << t) && !got[o]);
            got[o] = 1;
            V[tid * kRegs + i] = lds[o];
        }
}

// The program as fused.hip packs it (program_layout): phases, ops and
// coefficients, each part 256-byte aligned, 256 bytes behind the last.
struct Packed {
    size_t op_off, cf_off, total;
    explicit Packed(const Program& P) {
        const auto a256 = [](size_t x) { return (x + 255) & ~size_t(255); };
        op_off = a256(P.phases.size() * sizeof(FPhase));
        cf_off = a256(op_off + P.ops.size() * sizeof(FOp));
        total = cf_off + P.coef.size() * sizeof(double) + 256;
    }
};

struct Edge {
    bool own;
    uint32_t pos[kRegBits], global[kRegBits];
    Edge(const FPass& pass, int e, bool allow, unsigned rows) {
        own = allow && !pass.edge_dense[e] && byte_of(pass.edge[e], 0) >= rows;
        for (int j = 0; j < kRegBits; ++j) {
            pos[j] = own ? byte_of(pass.edge[e], j) : pass.t - kRegBits + j;
            global[j] = byte_of(own ? pass.edge_global[e] : pass.top_global, j);
        }
    }
};

static unsigned own_edges = 0, top_edges = 0, dense_edges = 0, permuted_passes = 0;

static void tile_pass(C* psi, uint64_t len, const Program& P, const FPass& pass, unsigned rows) {
    const uint32_t t = pass.t, nth = pass.nthreads;
    const Packed packed(P);
    CHECK(t >= 4 && t <= (uint32_t)kMaxTile && nth == 1u << (t - kRegBits));
    CHECK(pass.phase_begin < pass.phase_end && pass.phase_end <= P.phases.size());
    CHECK(pass.op_begin <= pass.op_end && pass.op_end <= P.ops.size());
    CHECK(pass.coef_begin <= pass.coef_end && pass.coef_end <= P.coef.size());
    // the edges' tables
    for (int e = 0; e < 2; ++e) {
        const FPhase& ph = P.phases[e ? pass.phase_end - 1 : pass.phase_begin];
        CHECK(pass.edge_dense[e] == ph.dense);
        for (int j = 0; j < kRegBits; ++j) {
            CHECK(ph.rpos[j] < t && byte_of(pass.edge[e], j) == ph.rpos[j]);
            CHECK(byte_of(pass.edge_global[e], j) == pass.tpos[ph.rpos[j]]);
            CHECK(byte_of(pass.top_global, j) == pass.tpos[t - kRegBits + j]);
        }
    }
    // one op and one phase ahead, across the pass's phases
    uint32_t o = pass.op_begin;
    const auto op_readable = [&](uint32_t k) { return packed.op_off + (k + 1) * sizeof(FOp) <= packed.total; };
    CHECK(op_readable(o));
    for (uint32_t p = pass.phase_begin; p < pass.phase_end; ++p) {
        const FPhase& ph = P.phases[p];
        CHECK((p + 2) * sizeof(FPhase) <= packed.total);
        CHECK(ph.op_begin == o && ph.op_end >= o && (!ph.dense || ph.op_end == o));
        if (ph.dense) {
            CHECK(ph.ucoef >= pass.coef_begin && ph.ucoef + 2 * kRegs * kRegs <= pass.coef_end);
        }
        o = ph.op_end;
        CHECK(op_readable(o));
    }
    CHECK(o == pass.op_end);

    const Edge in(pass, 0, true, rows), out(pass, 1, !pass.permuted, rows);
    (in.own ? own_edges : top_edges) += 1;
    (out.own ? own_edges : top_edges) += 1;
    dense_edges += pass.edge_dense[0] + pass.edge_dense[1];
    permuted_passes += pass.permuted;
    std::vector<C> V(nth * kRegs);
    std::vector<Layout> cur(nth);
    const auto global = [&](uint64_t tile, const Edge& e, uint32_t tb, int i) {
        uint64_t g = tile;
        for (uint32_t k = 0; k < t; ++k) g |= (uint64_t)(tb >> k & 1u) << pass.tpos[k];
        for (int j = 0; j < kRegBits; ++j)
            if (i >> j & 1) g += 1ull << e.global[j];
        CHECK(g < len);
        return g;
    };
    const auto own_offset = [&](uint64_t g, uint64_t tile) {  // local index of a global one
        uint32_t l = 0;
        for (uint32_t k = 0; k < t; ++k) l |= (uint32_t)(g >> pass.tpos[k] & 1u) << k;
        uint64_t back = tile;
        for (uint32_t k = 0; k < t; ++k) back |= (uint64_t)(l >> k & 1u) << pass.tpos[k];
        CHECK(back == g);
        return l;
    };
    for (uint64_t index = 0; index < len >> t; ++index) {
        uint64_t tile = index;
        for (uint32_t k = 0; k < t; ++k) {
            const uint64_t lo = tile & ((1ull << pass.tpos[k]) - 1u);
            tile = ((tile ^ lo) << 1) | lo;
        }
        std::vector<char> read(1u << t, 0), written(1u << t, 0);
        std::vector<uint32_t> tb(nth);
        for (uint32_t tid = 0; tid < nth; ++tid) {
            tb[tid] = spread(tid, in.pos);
            cur[tid] = layout_of(tb[tid], in.pos);
            for (int i = 0; i < kRegs; ++i) {
                const uint64_t g = global(tile, in, tb[tid], i);
                const uint32_t l = own_offset(g, tile);
                CHECK(!read[l] && tswz(l) == cur[tid](i));
                read[l] = 1;
                V[tid * kRegs + i] = psi[g];
            }
        }
        for (uint32_t p = pass.phase_begin; p < pass.phase_end; ++p) {
            const FPhase& ph = P.phases[p];
            if (ph.dense) {
                CHECK(t >= (uint32_t)kMinDenseTile);
                std::vector<Layout> to(nth);
                for (uint32_t tid = 0; tid < nth; ++tid) to[tid] = dense_layout(ph, tid);
                exchange(V, t, cur, [&](uint32_t tid, int i) { return to[tid](i); });
                cur = to;
                // register 4 c + s of lane l: row 4 s + l / 16, column 16 c + l % 16 of its wave
                for (uint32_t wave = 0; wave < nth / 64; ++wave) {
                    C X[kRegs][64];
                    for (uint32_t lane = 0; lane < 64; ++lane)
                        for (uint32_t c = 0; c < 4; ++c)
                            for (uint32_t s = 0; s < 4; ++s) {
                                const uint32_t row = 4 * s + lane / 16, col = 16 * c + lane % 16, tid = wave * 64 + lane;
                                uint32_t e = spread(wave * 64 + col, ph.rpos);
                                for (int j = 0; j < kRegBits; ++j)
                                    if (row >> j & 1) e |= 1u << ph.rpos[j];
                                CHECK(element(cur[tid]((int)(4 * c + s))) == e);
                                X[row][col] = V[tid * kRegs + 4 * c + s];
                            }
                    for (uint32_t lane = 0; lane < 64; ++lane)
                        for (uint32_t c = 0; c < 4; ++c)
                            for (uint32_t s = 0; s < 4; ++s) {
                                C acc = 0.0;
                                for (int k = 0; k < kRegs; ++k) acc += cf(P, ph.ucoef, (int)(4 * s + lane / 16) * kRegs + k) * X[k][16 * c + lane % 16];
                                V[(wave * 64 + lane) * kRegs + 4 * c + s] = acc;
                            }
                }
                continue;
            }
            if (p != pass.phase_begin || !(in.own || pass.direct_first)) {
                std::vector<Layout> to(nth);
                for (uint32_t tid = 0; tid < nth; ++tid) {
                    tb[tid] = spread(tid, ph.rpos);
                    to[tid] = layout_of(tb[tid], ph.rpos);
                }
                exchange(V, t, cur, [&](uint32_t tid, int i) { return to[tid](i); });
                cur = to;
            }
            for (uint32_t tid = 0; tid < nth; ++tid) {
                CHECK(tb[tid] == spread(tid, ph.rpos));
                for (int i = 0; i < kRegs; ++i) CHECK(cur[tid](i) == layout_of(tb[tid], ph.rpos)(i));
                run_phase(&V[tid * kRegs], ph, P, tb[tid], tile);
            }
        }
        if (pass.permuted) {
            CHECK(!out.own && !pass.direct_last);
            exchange(V, t, cur, [&](uint32_t tid, int i) {
                uint32_t s = 0;
                for (uint32_t k = 0; k + kRegBits < t; ++k)
                    if (tid >> k & 1) s ^= swz(pass.pimg[k]);  // (fusion.hpp's swizzle is its own inverse)
                return tswz(s) ^ tswz(swz(pass.pout[i]));
            });
        } else if (!out.own && !pass.direct_last) {
            exchange(V, t, cur, [&](uint32_t tid, int i) { return layout_of(spread(tid, out.pos), out.pos)(i); });
        } else {
            for (uint32_t tid = 0; tid < nth; ++tid)
                for (int i = 0; i < kRegs; ++i) CHECK(cur[tid](i) == layout_of(spread(tid, out.pos), out.pos)(i));
        }
        for (uint32_t tid = 0; tid < nth; ++tid)
            for (int i = 0; i < kRegs; ++i) {
                const uint64_t g = global(tile, out, spread(tid, out.pos), i);
                const uint32_t l = own_offset(g, tile);
                CHECK(!written[l]);
                written[l] = 1;
                psi[g] = V[tid * kRegs + i];
            }
    }
}

// the pass fields that same_steps does not compare
static bool same_edges(const std::vector<Step>& a, const std::vector<Step>& b) {
    for (size_t k = 0; k < a.size(); ++k)
        for (size_t i = 0; !a[k].plain && i < a[k].prog.passes.size(); ++i) {
            const FPass &u = a[k].prog.passes[i], &v = b[k].prog.passes[i];
            if (std::memcmp(u.edge, v.edge, sizeof u.edge) || std::memcmp(u.edge_global, v.edge_global, sizeof u.edge_global) ||
                std::memcmp(u.edge_dense, v.edge_dense, sizeof u.edge_dense) || u.top_global != v.top_global ||
                u.op_begin != v.op_begin || u.op_end != v.op_end || u.coef_begin != v.coef_begin || u.coef_end != v.coef_end)
                return false;
        }
    return true;
}

static void check_tiles(const std::vector<qvnt_gate>& gates, unsigned n, unsigned tq, unsigned dense, bool single_plain, unsigned amp_bytes,
                        std::mt19937_64& g) {
    std::vector<Step> steps, par;
    plan(gates.data(), gates.size(), n, tq, steps, dense, single_plain, false, amp_bytes);
    plan(gates.data(), gates.size(), n, tq, par, dense, single_plain, true, amp_bytes);
    CHECK(same_steps(steps, par) && same_edges(steps, par));
    orc_reg* ref = orc_reg_with_state(n, 0);
    const uint64_t len = orc_reg_len(ref);
    std::normal_distribution<double> nd;
    std::vector<C> psi(len);
    for (auto& z : psi) z = C(nd(g), nd(g));
    std::memcpy(orc_reg_psi(ref), psi.data(), len * sizeof(C));
    orc_reg_apply(ref, gates.data(), gates.size());
    for (const Step& st : steps) {
        if (st.plain) {
            orc_reg* one = orc_reg_with_state(n, 0);
            std::memcpy(orc_reg_psi(one), psi.data(), len * sizeof(C));
            orc_reg_apply(one, &st.gate, 1);
            std::memcpy(psi.data(), orc_reg_psi(one), len * sizeof(C));
            orc_reg_free(one);
            continue;
        }
        for (const FPass& fp : st.prog.passes) tile_pass(psi.data(), len, st.prog, fp, amp_bytes == 16 ? 3 : 4);
    }
    const C* want = reinterpret_cast<const C*>(orc_reg_psi(ref));
    double err = 0.0;
    for (uint64_t i = 0; i < len; ++i) err = std::max(err, std::abs(psi[i] - want[i]));
    std::printf("n=%u tq=%u dense=%u %u bytes: %zu gates, max |d| %.2e\n", n, tq, dense, amp_bytes, gates.size(), err);
    if (!(err <= 1e-12)) ++failures;
    orc_reg_free(ref);
}

int main() {
    uint64_t seed = 100;
    for (unsigned bytes : {16u, 8u}) {
        const unsigned cases[][3] = {{6, 6, 0}, {7, 6, 0}, {9, 8, 0}, {10, 10, 2}, {11, 9, 0}, {12, 12, 3}, {13, 12, 2}, {14, 10, 2}, {15, 11, 0}, {15, 12, 4}};
        for (const auto& c : cases) {
            std::mt19937_64 g(seed++);
            check_tiles(random_circuit(g, c[0], 160), c[0], c[1], c[2], false, bytes, g);
        }
        const unsigned layered[][3] = {{10, 10, 0}, {13, 12, 0}, {14, 11, 0}, {16, 12, 3}};
        for (const auto& c : layered) {
            std::mt19937_64 g(seed++);
            check_tiles(layered_circuit(g, c[0], 5), c[0], c[1], c[2], true, bytes, g);
        }
    }
    {
        std::mt19937_64 g(seed++);
        check_tiles(random_circuit(g, 15, 200), 15, 13, 3, false, 8, g);  // FP32's largest tile
        check_tiles(cx_high_layer(g, 17), 17, 11, 0, false, 16, g);
    }
    std::printf("edges: %u own, %u top, %u dense; %u permuted passes\n", own_edges, top_edges, dense_edges, permuted_passes);
    if (!own_edges || !top_edges || !dense_edges || !permuted_passes) ++failures;
    std::printf("%d failure(s)\n", failures);
    return failures ? 1 : 0;
}
