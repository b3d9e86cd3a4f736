// plan_resident.cpp -- the resident time loop of a plan (psv_resident.inc): when it is
// used, the partition of the grid into tiles, the point tables and the launch.
#include <type_traits>

#include "plan.h"

namespace psvplan {

namespace {

// The rows of one column of tiles.  A tile is interior when the rows it owns are in
// [zlo, zhi) (and xin, the same in x).  Interior tiles take up to `own` rows, edge tiles up to
// `own_edge`; the fewest tiles that cover the column.  The columns they cover are the caller's.
std::vector<psv::ResTile> tile_column(int nzt, int zlo, int zhi, bool xin, int own, int own_edge)
{
    std::vector<psv::ResTile> out;
    // need[z]: tiles for the rows from z on; step[z]: height of the first, negative for interior
    std::vector<int> need((size_t)nzt + 1, 0), step((size_t)nzt + 1, 0);
    for (int z = nzt - 1; z >= 0; z--) {
        const int he = std::min(own_edge, nzt - z);
        need[(size_t)z] = 1 + need[(size_t)(z + he)];
        step[(size_t)z] = he;
        const int hi = std::min(own, zhi - z);
        if (xin && z >= zlo && hi > 0 && 1 + need[(size_t)(z + hi)] <= need[(size_t)z]) {
            need[(size_t)z] = 1 + need[(size_t)(z + hi)];
            step[(size_t)z] = -hi;
        }
    }
    for (int z = 0; z < nzt;) {
        const int h = step[(size_t)z] < 0 ? -step[(size_t)z] : step[(size_t)z];
        psv::ResTile t{};
        t.z0 = z;
        t.z1 = z + h;
        t.zr = std::max(0, z - psv::kResHalo);
        t.edge = step[(size_t)z] < 0 ? 0 : 1;
        out.push_back(t);
        z += h;
    }
    return out;
}

}  // namespace

// The tiles of the grid for a shape, in strips of at most `cap` (none: they do not fit).
// Interior tiles: every stress cell they compute (2 cells around the owned ones) is updated, outside the CPML strips and below the free-surface row; for the transposed steps also
// every velocity weight they form (kResHalo cells around) is one of an updated cell outside the
// strips, and none of their stress cells is mirrored.
template <typename T>
typename Plan<T>::Partition Plan<T>::resident_tiles(const psv::ResShape& sh, bool discrete, int most_rows, int cap) const
{
    const int nzt = g_.nzt, nxt = g_.nxt, H = fpad_;
    const bool pml = g_.npml > 0;
    int zlo = 2 + (g_.fsurf ? H + 1 : (pml ? ppad_ + 1 : H));
    int zhi = (pml ? nzt - ppad_ - 1 : nzt - H) - 2;
    int xlo = 2 + (pml ? ppad_ + 1 : H), xhi = (pml ? nxt - ppad_ - 1 : nxt - H) - 2;
    if (discrete) {
        zlo = std::max(zlo, g_.fsurf ? 2 * H + 3 : psv::kResHalo + (pml ? ppad_ : H));
        xlo = std::max(xlo, psv::kResHalo + (pml ? ppad_ : H));
        zhi -= psv::kResHalo - 2;
        xhi -= psv::kResHalo - 2;
    }
    const int own = std::min(sh.rows * sh.waves - 2 * psv::kResHalo, most_rows);
    const int own_edge = std::min(sh.rows_edge * sh.waves - 2 * psv::kResHalo, most_rows);
    // a column's rows depend on whether it is an inner one: formed once, so that a partition that
    // does not fit is only counted (1084 x 584: the first pass of a plan 5.5 -> 1.3 ms over the next)
    const std::vector<psv::ResTile> rows_of[2] = {tile_column(nzt, zlo, zhi, false, own, own_edge),
                                                  tile_column(nzt, zlo, zhi, true, own, own_edge)};
    auto column = [&](int x0, int x1) -> const std::vector<psv::ResTile>& { return rows_of[x0 >= xlo && x1 <= xhi]; };
    // columns: the first and last tile have a halo on one side only
    const int W = psv::kResOwnX, end = W + psv::kResHalo;
    const int ncol = nxt <= 64 ? 1 : (nxt <= 2 * end ? 2 : 2 + (nxt - 2 * end + W - 1) / W);
    std::vector<int> cx(1, 0);
    for (int c = 0, x = 0; c < ncol; c++) {
        // even widths, within what each column can hold
        const int left = ncol - 1 - c, rest = left == 0 ? 0 : (left - 1) * W + end;
        const int most = ncol == 1 ? 64 : (c == 0 || left == 0 ? end : W);
        const int x1 = x + std::min(most, std::max((nxt - x + left) / (left + 1), nxt - x - rest));
        cx.push_back(x1);
        x = x1;
    }
    // f(x0, x1, shadow, xs, xe) for the columns of strip k of n, its own and then `around` on each side
    auto strip = [&](int k, int n, int around, auto f) {
        const int c0 = k * ncol / n, c1 = (k + 1) * ncol / n, ext = around * psv::kStripCells;
        const int xa = cx[(size_t)c0], xb = cx[(size_t)c1];
        const int xs = std::max(0, xa - ext), xe = std::min(nxt, xb + ext);
        for (int c = c0; c < c1; c++) f(cx[(size_t)c], cx[(size_t)c + 1], 0, xs, xe);
        for (int x = xa; x > xs; x -= psv::kStripCells) f(std::max(xs, x - psv::kStripCells), x, 1, xs, xe);
        for (int x = xb; x < xe; x += psv::kStripCells) f(x, std::min(xe, x + psv::kStripCells), 1, xs, xe);
    };
    // the fewest strips of even numbers of columns, then the most columns around each
    for (int n = 1; n <= ncol; n++)
        for (int around = n == 1 ? 1 : psv::kStripColumns; around >= 1; around--) {
            bool fits = true;
            for (int k = 0; k < n && fits; k++) {
                int tiles = 0;
                strip(k, n, around, [&](int x0, int x1, int, int, int) { tiles += (int)column(x0, x1).size(); });
                fits = tiles <= cap;
            }
            if (!fits) continue;
            Partition p;
            p.strips.assign(1, 0);
            p.steps = around * psv::kStripSteps;
            int rows = 0;
            for (int k = 0; k < n; k++) {
                strip(k, n, around, [&](int x0, int x1, int shadow, int xs, int xe) {
                    for (psv::ResTile t : column(x0, x1)) {
                        t.x0 = x0;
                        t.x1 = x1;
                        t.xr = std::max(0, x0 - psv::kResHalo);
                        t.xs = xs;
                        t.xe = xe;
                        t.shadow = shadow;
                        t.row0 = rows;
                        if (!shadow) rows += sh.waves * (t.edge ? sh.rows_edge : sh.rows);
                        p.h.push_back(t);
                    }
                });
                p.strips.push_back((int)p.h.size());
            }
            return p;
        }
    return Partition();
}

// A split step of `n` shots in us: two launches that a small grid does not fill, then the
// bytes it moves.  Fitted to one MI355X (order 4, forward and adjoint mean): FP32 12.7 on
// 55 k cells, 17.3 on 0.63 M, 25 on 1.08 M and 25 on 16 x 52 k; FP64 15 on 0.2 M, 28 on
// 0.63 M, 38 on 0.82 M; compensated FP32 20 on 55 k and 21 on 0.2 M.
static double split_step_us(double cells, int esize, bool dwords)
{
    const double floor = dwords ? 20.0 : 12.5;
    return std::max(floor, 5.0 + cells * (esize == 4 ? 19e-6 : 39e-6));
}

// What a strip's launch of some steps takes besides them, per step: the launch, ten arrays in and
// five out.  (Half of 2484 x 884 in FP32: 20 us between the launches and 20 us of each.)
static double strip_move_us(double cells, int esize, int steps)
{
    return (20.0 + cells * 15 * esize / 4e6) / steps;
}

// The forward and the adjoint step apart.  Split, us a step of `cells` M cells: FP32 forward 11.1 on
// 0.06, 16.3 on 0.63, 38 on 2.2, 73 on 4.7, 154 on 9.6, 478 on 28, adjoint 11.7, 17.8, 45, 87, 207, 575;
// FP64 forward 13.8 on 0.008, 31 on 0.81, 65 on 2.2, 154 on 4.7, 370 on 10.6, adjoint 14.0, 36, 79, 206,
// 438 (above 2 to 7 M the arrays no longer fit in the Infinity Cache); compensated FP32 18 on 0.06, 34 on
// 0.45.
static double split_us(double cells, int esize, bool dwords, bool forward)
{
    if (dwords) return 16.5 + 38.0 * cells;
    if (esize == 4) {
        const double us = forward ? 9.0 + 12.9 * cells + 4.1 * std::max(0.0, cells - 7.0)
                                  : 9.0 + 17.0 * cells + 4.0 * std::max(0.0, cells - 5.0);
        return std::max(11.0, us);
    }
    const double over = std::max(0.0, cells - 2.2);
    return forward ? 12.0 + 23.5 * cells + 12.5 * over : 12.0 + 31.0 * cells + 11.0 * over;
}

// A launch of the resident loop besides its steps, us, where its tiles have `cells` M cells: it
// starts, loads the state and the model and writes the state back.  Measured FP32 forward 21 on 0.06,
// 28 on 0.63, 40 on 1.08, and a strip's 43 on 1.4, 50 on 1.6, adjoint 21, 37, 54, 72, 80; FP64 forward
// 27 on 0.26, 36 on 0.41, a strip's 51 on 0.85, adjoint 32, 46, 66.
static double launch_us(double cells, int esize, bool forward)
{
    return 20.0 + cells * esize / 4 * (forward ? (esize == 4 ? 17.0 : 20.0) : (esize == 4 ? 36.0 : 25.0));
}

// Launches of a resident run of `steps` steps, per strip: one, or an even number.
template <typename T>
int Plan<T>::resident_parts(int steps) const
{
    if (res_.part.strips.size() <= 2) return 1;
    const int parts = (steps + res_.part.steps - 1) / res_.part.steps;
    return steps > 1 ? parts + (parts & 1) : parts;
}

// Whether the resident loop pays in a run of records or segments of `steps` steps that are run
// forward, backward or (the replay of a segment) both; resident_ready's choice is by the mean of a
// forward and an adjoint step over a long run.  A strip's launches are half a segment long at most.
// The line lies where the two sums meet: 8 steps of 3600 x 1200 in FP32, forward, 0.61 ms resident
// and 0.55 split (12 steps 0.71, 0.81); checkpoints 8 apart there, replay and adjoint of 96 steps,
// 19.4 and 16.2 ms (12 apart 15.1, 16.1); 600 x 300 in FP64, adjoint, 2 steps 0.059 and 0.054
// (3 steps 0.060, 0.074); 2000 x 4000 in FP64, where the adjoint step of the largest tiles spills,
// forward 244 us a step and 298, adjoint 459 and 353.
template <typename T>
bool Plan<T>::resident_for(int steps, bool forward, bool adjoint, bool grad)
{
    constexpr bool dwords = std::is_same<T, psv::dfloat>::value;
    constexpr int esize = (int)sizeof(T);
    // (the split step's tiles are 64 columns wide: half a column beyond the grid costs what one in it does)
    const double all = 1e-6 * nslots_ * g_.nzt * (g_.nxt + (double)round_up((size_t)g_.nxt, 64)) / 2;
    double split = 0, least = 0;
    for (bool f : {true, false})
        if (f ? forward : adjoint) {
            split += split_us(all, esize, dwords, f);
            least += 2.9 + launch_us(all, esize, f) / steps;
        }
    // (no search for a shape where none could pay)
    if (least >= split || !resident_ready()) return false;
    const int parts = resident_parts(steps);
    double cost = 0;
    for (bool f : {true, false})
        if (f ? forward : adjoint)
            cost += res_.rounds * (res_.us[f ? 0 : (grad ? 1 : 2)] + launch_us(res_.cells, esize, f) * parts / steps);
    return cost < split && resident_alloc();
}

// The same for the exact gradient's segments of `steps` steps, replay and transposed steps.  Resident,
// the two take about 2.8 forward steps (us a step of a strip: FP32 12 x 9 rows 21.5, FP64 8 x 6 17.5,
// 8 x 9 46) and their launches 40 us and 62 a M cells of FP32; split, us a step: FP32 28 on 0.06 M cells,
// 61 on 0.63, 180 on 2.8, 300 on 4.7, 580 on 9.6, FP64 30 on 0.008, 280 on 2.2, 1050 on 8.5, compensated
// FP32 42 on 0.06.  The line: 2000 x 4000 in FP64, segments of 8 steps 1490 us a step and 1110, of 32
// 1000 and 1070; 1500 x 6000 in FP32, of 8 710 and 600, of 16 500 and 600.
template <typename T>
bool Plan<T>::resident_exact(int steps)
{
    if (!resident_ready() || !res_.discrete) return false;
    constexpr int esize = (int)sizeof(T);
    const double all = 1e-6 * nslots_ * g_.nzt * g_.nxt;
    const double split = esize == 4 ? 25.0 + 57.0 * all : (std::is_same<T, psv::dfloat>::value ? 38.0 : 28.0) + 118.0 * all;
    const double launch = 40.0 + 62.0 * res_.cells * esize / 4;
    return res_.rounds * (2.8 * res_.us_mean + launch * resident_parts(steps) / steps) < split && resident_alloc();
}

// Whether the plan's runs can take the resident loop, and its shape for the current batch.
// Not for a caller who chose a tile height; not for CPML profiles that couple the strips
// (the reference's arrays give the innermost cells of the two strips of an axis one memory
// cell, which stays zero only while a = a_half = 0 there), nor for grids whose strips meet.
template <typename T>
bool Plan<T>::resident_ready()
{
    const psv::ResShape* shapes = nullptr;
    const int n = psv::resident_shapes<T>(&shapes);
    if (n == 0 || !tile_auto_ || res_.failed || nslots_ < 1) return false;
    if (g_.npml > 0) {
        if (!have_pml_ || h_pml_[(size_t)g_.npml] != 0.0 || h_pml_[(size_t)3 * tp_ + g_.npml] != 0.0) return false;
        if (g_.nxt - 2 * ppad_ < 3 || g_.nzt - 2 * ppad_ < 3) return false;
    }
    // every tile needs room for the mirror rows and the rim of a neighbour
    if (g_.nxt < 16 || g_.nzt < 16) return false;
    // the exchange buffer is addressed in 32 bits
    if ((double)(g_.nzt + 8) * (g_.nxt + 8) * 8 * sizeof(T) >= 2147483648.0) return false;
    const bool want = grad_mode_ == PSVFWI_GRADIENT_DISCRETE;
    if (res_.slots == nslots_ && res_.want == want) return res_.shape >= 0;
    res_.slots = nslots_;
    res_.want = want;
    res_.shape = -1;
    // with the exact gradient, a shape that has the replay and the reverse steps; without one,
    // a shape for the forward runs only
    for (int d = want; d >= 0 && res_.shape < 0; d--) {
        // the shots run conc at a time, rounds times over; the split step takes them together
        double best = split_step_us((double)nslots_ * g_.nzt * g_.nxt, (int)sizeof(T), std::is_same<T, psv::dfloat>::value);
        for (int i = 0; i < n; i++) {
            int cap = 1 << 30;
            for (int mode = psv::kForward; mode <= (d ? psv::kReverse : (int)psv::kAdjoint); mode++) {
                int c = 0;
                if (psv::resident_capacity<T>(g_.fdorder, mode, i, &c) != hipSuccess) c = 0;
                cap = std::min(cap, c);
            }
            const Partition p = resident_tiles(shapes[i], d != 0, g_.nzt, cap);
            if (p.h.empty()) continue;
            const int ns = (int)p.strips.size() - 1;
            const int conc = ns > 1 ? 1 : std::min(nslots_, cap / (int)p.h.size());
            // launches a step, and what starting one and moving its state adds to a step of a strip
            const int rounds = ns > 1 ? nslots_ * ns : (nslots_ + conc - 1) / conc;
            const double move = ns > 1 ? strip_move_us((double)g_.nzt * g_.nxt / ns, (int)sizeof(T), p.steps) : 0.0;
            const double cost = rounds * (shapes[i].us + move);
            if (cost < best) {
                best = cost;
                res_.us_mean = shapes[i].us;
                res_.us[0] = shapes[i].forward;
                res_.us[1] = shapes[i].adjoint;
                // without the correlation (2000 x 4000 in FP64, largest tiles: 338 us a step for 459)
                res_.us[2] = (2 * shapes[i].forward + shapes[i].adjoint) / 3;
                res_.rounds = rounds;
                res_.shape = i;
                res_.conc = conc;
                res_.cap = cap;
                res_.part = p;
                res_.discrete = d != 0;
            }
        }
    }
    (void)hipGetLastError();  // a shape that is not built is no error
    if (res_.shape < 0) return false;
    // a grid that needs fewer workgroups than there are CUs takes lower tiles: waves without
    // rows to compute leave their SIMD to the others (down to 6 rows, where a shape's two rows a
    // wave are still shared evenly; 241 x 221, 190 tiles for 115, a step: compensated FP32
    // 10.4 -> 9.0 us, FP32 and FP64 3 % less)
    for (int own = 6; own < g_.nzt; own++) {
        const Partition p = resident_tiles(shapes[res_.shape], res_.discrete, own, res_.cap / res_.conc);
        if (!p.h.empty() && p.strips.size() == res_.part.strips.size() && p.steps == res_.part.steps) {
            res_.part = p;
            break;
        }
    }
    res_.cells = 0;
    for (const psv::ResTile& t : res_.part.h) res_.cells += (double)(t.z1 - t.z0) * (t.x1 - t.x0);
    res_.cells *= 1e-6 * (res_.part.strips.size() > 2 ? 1.0 / (res_.part.strips.size() - 1) : res_.conc);
    res_.waves = shapes[res_.shape].waves;
    res_.rows = shapes[res_.shape].rows;
    res_.rows_edge = shapes[res_.shape].rows_edge;
    res_.gen++;
    res_.uploaded = false;
    return true;
}

// The memory of the chosen tiles, for a run that takes the loop: the exchange buffer, the flag, and
// for strips the other set of a slot's state; false (and no loop for this batch) where there is none.
template <typename T>
bool Plan<T>::resident_alloc()
{
    if (res_.alloc_gen == res_.gen) return true;
    res_.xpitch = (int)round_up((size_t)g_.nxt, 8);
    res_.zpitch = (int)round_up((size_t)g_.nzt, 8);
    res_.exch_slot = 2 * ((size_t)g_.nzt * res_.xpitch + (size_t)g_.nxt * res_.zpitch) * (2 * sizeof(T) / 4);
    const size_t need = res_.exch_slot * (size_t)res_.conc;
    bool ok = true;
    if (!res_.exch.p || res_.exch.cap < need) {
        ok = res_.exch.alloc(need) == hipSuccess &&
             psv::launch_fill<unsigned long long>(res_.exch.p, need, 0ull, stream_) == hipSuccess;
        res_.tag = 1;
    }
    if (ok && !res_.aborted) {
        ok = hipHostMalloc(reinterpret_cast<void**>(&res_.aborted), sizeof(int), hipHostMallocMapped) == hipSuccess;
        if (ok) *res_.aborted = 0;
    }
    const bool two = res_.part.strips.size() > 2;
    for (int k = 0; k < psv::kStateArrays && ok && two; k++) {
        const size_t n = k < 5 ? fst_ : (g_.npml > 0 ? (k < 9 ? xst_ : zst_) : 0);
        ok = res_.other[k].alloc(n) == hipSuccess && (n == 0 || psv::launch_fill<T>(res_.other[k].p, n, (T)0, stream_) == hipSuccess);
    }
    if (!ok) {
        (void)hipGetLastError();
        for (DBuf<T>& b : res_.other) b.release();
        res_.exch.release();
        res_.shape = -1;
        return false;
    }
    res_.alloc_gen = res_.gen;
    return true;
}

// the point tables of a Tables object for the current tiles (ResPoints)
template <typename T>
psvfwi_status Plan<T>::resident_points(Tables& t)
{
    if (t.res_gen == res_.gen) return PSVFWI_OK;
    const int ntile = (int)res_.part.h.size();
    const int nw = res_.waves;
    struct Layer {
        int head;
        std::vector<int> id;
    };
    std::vector<std::vector<Layer>> lay((size_t)nslots_ * ntile * nw);
    // entry `v` of component `comp` at (z, x): the first layer of its wave, row and component
    // whose lane is free, so that entries of one cell keep their order
    auto add = [&](int slot, int k, int z, int x, int comp, int rec, int v) {
        const psv::ResTile& q = res_.part.h[(size_t)k];
        const int R = q.edge ? res_.rows_edge : res_.rows;
        const int row = z - q.zr, lane = x - q.xr;
        std::vector<Layer>& l = lay[((size_t)slot * ntile + k) * nw + (size_t)(row / R)];
        const int head = (row % R) | comp << 8 | rec << 16;
        for (Layer& y : l)
            if (y.head == head && y.id[(size_t)lane] < 0) {
                y.id[(size_t)lane] = v;
                return;
            }
        l.push_back(Layer{head, std::vector<int>(64, -1)});
        l.back().id[(size_t)lane] = v;
    };
    for (int s = 0; s < nslots_; s++)
        for (int rec = 0; rec < 2; rec++) {
            const std::vector<int>& off = rec ? t.rec_off : t.grp_off;
            for (int g = off[(size_t)s]; g < off[(size_t)s + 1]; g++) {
                const int* e = rec ? &t.zxc_h[3 * (size_t)g] : &t.grp_h[5 * (size_t)g];
                const int z = e[0], x = e[1], comp = e[2];
                for (int k = 0; k < ntile; k++) {
                    const psv::ResTile& q = res_.part.h[(size_t)k];
                    // stress sources act on the stresses a tile computes around its own cells too
                    const int ring = !rec && comp == 4 ? 2 : 0;
                    if (z < q.z0 - ring || z >= q.z1 + ring || x < q.x0 - ring || x >= q.x1 + ring) continue;
                    if (rec && q.shadow) continue;
                    if (rec) add(s, k, z, x, comp, 1, g - off[(size_t)s]);
                    else
                        for (int j = 0; j < e[4]; j++) add(s, k, z, x, comp, 0, t.row_h[(size_t)(e[3] + j)]);
                }
            }
        }
    std::vector<int> off(lay.size() + 1, 0), head, id;
    for (size_t i = 0; i < lay.size(); i++) {
        off[i + 1] = off[i] + (int)lay[i].size();
        for (const Layer& y : lay[i]) {
            head.push_back(y.head);
            id.insert(id.end(), y.id.begin(), y.id.end());
        }
    }
    PSV_HIP(t.res_off.alloc(off.size()));
    PSV_HIP(t.res_head.alloc(std::max<size_t>(head.size(), 1)));
    PSV_HIP(t.res_id.alloc(std::max<size_t>(id.size(), 64)));
    PSV_HIP(hipMemcpy(t.res_off.p, off.data(), off.size() * sizeof(int), hipMemcpyHostToDevice));
    if (!head.empty()) {
        PSV_HIP(hipMemcpy(t.res_head.p, head.data(), head.size() * sizeof(int), hipMemcpyHostToDevice));
        PSV_HIP(hipMemcpy(t.res_id.p, id.data(), id.size() * sizeof(int), hipMemcpyHostToDevice));
    }
    t.res_gen = res_.gen;
    return PSVFWI_OK;
}

// the tiles of the resident loop and the point tables of a run, on the device before its timed part
template <typename T>
psvfwi_status Plan<T>::resident_prepare(std::initializer_list<Tables*> tabs)
{
    // (a run that ended with another error may have left it set; set before a run, waits are over
    // after their first look at it)
    *res_.aborted = res_.mute == 1;
    if (!res_.uploaded || res_.mute) {
        std::vector<psv::ResTile> h = res_.part.h;
        // a tile at the edge of a strip has no neighbour there
        if (res_.mute) h[0].xe = h[0].x1;
        PSV_HIP(res_.tiles.alloc(h.size()));
        PSV_HIP(hipMemcpy(res_.tiles.p, h.data(), h.size() * sizeof(psv::ResTile), hipMemcpyHostToDevice));
        res_.uploaded = res_.mute == 0;
    }
    for (Tables* t : tabs) PSV_TRY(resident_points(*t));
    return PSVFWI_OK;
}

// Steps [it0, it1) of the current launch group in one launch: forward in time, or for the
// adjoint backward from each shot's min(it1, nt) - 1.
template <typename T>
psvfwi_status Plan<T>::launch_resident(State<T>& st, Tables& tab, bool fwd_sig, int mode, int kind, int it0, int it1,
                                       int flags, int tf0, bool one_plane)
{
    const int steps = it1 - it0;
    psv::ResidentParams<T> a{};
    if (mode >= psv::kReplay) {
        a.terms = seg_.p;
        a.terms_slot = resident_terms();
        a.terms_step = a.terms_slot * (size_t)res_.conc;
        a.terms_it0 = it0;
        for (int i = 0; i < 5; i++) a.g5[i] = atw(dg_[i], fst_);
    }
    a.p = base_params(st, tab, fwd_sig);
    a.p.nslots = active(it0);
    a.p.flags = flags;
    a.p.tf0 = tf0;
    a.pts.head = tab.res_head.p;
    a.pts.id = tab.res_id.p;
    a.tf_stride = one_plane ? 0 : (size_t)5 * nfz_ * nfx_;
    a.exch = res_.exch.p;
    a.exch_slot = res_.exch_slot;
    a.xpitch = res_.xpitch;
    a.zpitch = res_.zpitch;
    a.aborted = res_.aborted;
    a.kdiv = res_.kdiv;
    T** const in[psv::kStateArrays] = {&a.p.vx, &a.p.vz, &a.p.sxx, &a.p.szx, &a.p.szz, &a.p.mvxx, &a.p.mvzx,
                                       &a.p.msxxx, &a.p.mszxx, &a.p.mvzz, &a.p.mvxz, &a.p.mszzz, &a.p.mszxz};
    const int nstrip = (int)res_.part.strips.size() - 1;
    for (int k = 0; k < psv::kStateArrays; k++) a.out[k] = nstrip > 1 ? res_.other[k].p + (k < 5 ? org_ : 0) : *in[k];
    const bool sample = kind >= 0 && sample_ev_[0][0] && nsamp_ < kMaxSamples;
    if (sample) PSV_HIP(hipEventRecord(sample_ev_[nsamp_][0], stream_));
    // one launch of all steps; strips (one slot at a time): an even number of launches of a few
    // steps each, which ends in the slot's own arrays, each writing the other set of the state
    const int last = nstrip > 1 ? std::min(it1, group_nt()) : it1, n = last - it0;
    const int parts = resident_parts(n);
    hipError_t e = hipSuccess;
    for (int j = 0; j < parts && e == hipSuccess; j++) {
        const bool back = mode == psv::kAdjoint || mode == psv::kReverse;
        const int b0 = (int)((long long)n * j / parts), b1 = (int)((long long)n * (j + 1) / parts);
        a.it0 = back ? last - b1 : it0 + b0;
        a.it1 = back ? last - b0 : it0 + b1;
        if (nstrip == 1) a.it1 = it1;
        const unsigned span = (unsigned)(a.it1 - a.it0);
        for (int k = 0; k < nstrip && e == hipSuccess; k++) {
            if (res_.tag > 0xffffffffu - span - 2u) {
                PSV_HIP(psv::launch_fill<unsigned long long>(res_.exch.p, res_.exch.cap, 0ull, stream_));
                res_.tag = 1;
            }
            const int t0 = res_.part.strips[(size_t)k];
            a.tiles = res_.tiles.p + t0;
            a.ntile = res_.part.strips[(size_t)k + 1] - t0;
            a.pts.off = tab.res_off.p + ((size_t)w0_ * res_.part.h.size() + (size_t)t0) * res_.waves;
            a.tag = res_.tag;
            res_.tag += span;
            if (res_.refuse > 0) {
                res_.refuse--;
                e = hipErrorCooperativeLaunchTooLarge;
            } else {
                e = psv::launch_resident<T>(a, g_.fdorder, mode, res_.shape, stream_);
            }
        }
        if (nstrip > 1)
            for (int k = 0; k < psv::kStateArrays; k++) std::swap(*in[k], a.out[k]);
    }
    // (a single step ends in the other set)
    for (int k = 0; nstrip > 1 && (parts & 1) && k < psv::kStateArrays && e == hipSuccess; k++)
        if (res_.other[k].n > 0)
            e = hipMemcpyAsync(a.out[k] - (k < 5 ? org_ : 0), res_.other[k].p, res_.other[k].n * sizeof(T),
                               hipMemcpyDeviceToDevice, stream_);
    if (e != hipSuccess) {
        // refused (no cooperative launch here): the caller runs the split step instead
        (void)hipGetLastError();
        *res_.aborted = 1;
        return PSVFWI_OK;
    }
    if (sample) {
        PSV_HIP(hipEventRecord(sample_ev_[nsamp_][1], stream_));
        samp_kind_[nsamp_] = kind;
        samp_steps_[nsamp_] = steps;
        samp_one_[nsamp_] = true;
        nsamp_++;
    }
    if (kind >= 0) launches_ += steps;
    return PSVFWI_OK;
}

// Elements of one step's derivative terms of a slot.
template <typename T>
size_t Plan<T>::resident_terms() const
{
    size_t rows = 0;
    for (const psv::ResTile& t : res_.part.h)
        if (!t.shadow) rows = std::max(rows, (size_t)t.row0 + res_.waves * (t.edge ? res_.rows_edge : res_.rows));
    return rows * 320;
}

// After the stream has drained: a resident run whose waits ran out, or that was refused,
// has left the state unusable; the plan then keeps to the split step and the run starts over.
template <typename T>
bool Plan<T>::resident_failed()
{
    if (!res_.aborted || *res_.aborted == 0) return false;
    *res_.aborted = 0;
    res_.failed = true;
    return true;
}

// For tests: the first tile sends nothing to its right, so that the tiles there wait in vain (mute 1:
// until their first look at `aborted`, 2: until they give up), the tag of the next launch (only up:
// the exchange buffer holds the ones before it), and how many launches are refused.
template <typename T>
psvfwi_status Plan<T>::test_resident(int mute, unsigned tag, int refuse)
{
    res_.mute = mute;
    res_.tag = std::max(res_.tag, tag);
    res_.refuse = refuse;
    return PSVFWI_OK;
}

#define PSV_INSTANTIATE(T) \
    template psvfwi_status Plan<T>::test_resident(int, unsigned, int); \
    template Plan<T>::Partition Plan<T>::resident_tiles(const psv::ResShape&, bool, int, int) const; \
    template bool Plan<T>::resident_ready(); \
    template bool Plan<T>::resident_for(int, bool, bool, bool); \
    template bool Plan<T>::resident_exact(int); \
    template int Plan<T>::resident_parts(int) const; \
    template bool Plan<T>::resident_alloc(); \
    template size_t Plan<T>::resident_terms() const; \
    template psvfwi_status Plan<T>::resident_points(Tables&); \
    template psvfwi_status Plan<T>::resident_prepare(std::initializer_list<Tables*>); \
    template psvfwi_status Plan<T>::launch_resident(State<T>&, Tables&, bool, int, int, int, int, int, int, bool); \
    template bool Plan<T>::resident_failed();
PSV_FOR_EACH_PRECISION(PSV_INSTANTIATE)

}  // namespace psvplan
