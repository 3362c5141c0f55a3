// tile3.hpp -- one 16^3 tile (plus its +1 halo) of a 3-D field on one
// workgroup of 256 lanes: the tile in LDS, the stages of the four levels, and
// the codes between the level-major array (or the bit-planes) and the tile.
//
// Reference: InterpolationPredictor.cu -- 1-D rule 1229-1352,
// multi-dimensional rule 1414-1750, level loop 1823-2026, tile staging
// 997-1170, compaction 2028-2088.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "spline_rules.hpp"

namespace pa {
namespace {

// ------------------------------------------------------------ LDS layout --
// Value (x, y, z) of the tile lies at z * 297 + Y(y) * 17 + x, where Y lists
// the even y before the odd ones.  A stage's lanes enumerate every other
// coordinate, which in the plain [17][17][17] order hit few of the banks:
// the multi-dimensional stages of a float32 tile took 7.2 LDS cycles per
// instruction, 5.1 of them conflicts.  The order, the plane pitch and the
// stages' lane enumerations were chosen together by counting the conflicts
// of every access of a level-0 pass (cycles of float32 / float64, forward
// + reverse + multi-dimensional: 5019 / 5519 plain, 3196 / 4724 here; all
// eight subsets of axes and pitches 289..301 were counted).  The strides
// along an axis stay compile-time constants, and 5041 values still let 4
// float64 or 8 float32 workgroups share the 160 KB.
constexpr int kYP = 17, kYO = 9 * 17, kZP = 297;
constexpr int kTileLds = 16 * kZP + 17 * 17;  // 5041

__host__ __device__ constexpr int tslot(int x, int y, int z) { return z * kZP + (y >> 1) * kYP + (y & 1) * kYO + x; }

// Along axis A (0 = x, 1 = y, 2 = z) at unit U: slots between even multiples
// of U (2U apart), and from an even multiple to the odd one after it.
template <int U, int A>
constexpr int slot_step() {
    return A == 0 ? 2 * U : (A == 1 ? U * kYP : 2 * U * kZP);
}
template <int U, int A>
constexpr int slot_half() {
    return A == 0 ? U : (A == 1 ? (U == 1 ? kYO : U / 2 * kYP) : U * kZP);
}

// IN: not the last tile along any axis, all 17^3 points inside the field
// (every stencil then is decided at compile time).  rx, ry, rz: points of the
// tile inside the field along each axis, halo included (17: not the last).
template <typename T, bool IN>
struct Tile {
    T* s;
    int ox, oy, oz;
    int rx, ry, rz;
    Geom g;
    T eb_r, ebx2;  // of the current level
    int32_t* qc_out;

    template <int A>
    __device__ __forceinline__ bool in(int c) const {
        return IN || c < (A == 0 ? rx : (A == 1 ? ry : rz));
    }
    __device__ __forceinline__ bool in3(int x, int y, int z) const { return IN || (x < rx && y < ry && z < rz); }
};

template <typename T, bool IN>
__device__ __forceinline__ Tile<T, IN> make_tile(const Geom& g, T* s, int bx, int by, int bz, int32_t* qc_out) {
    Tile<T, IN> t;
    t.s = s;
    t.ox = bx * 16;
    t.oy = by * 16;
    t.oz = bz * 16;
    t.rx = min(g.nx - t.ox, kTS);
    t.ry = min(g.ny - t.oy, kTS);
    t.rz = min(g.nz - t.oz, kTS);
    t.g = g;
    t.qc_out = qc_out;
    return t;
}

// ---------------------------------------------------------------- stencils --
// Point j of a line of N = 8 / U points lies between the known values j and
// j + 1 of N + 1 (0 .. last inside the field, last = N away from the far
// face).  Which neighbours exist decides its formula
// (InterpolationPredictor.cu:1269-1326, 1538-1545), in the order of
// preference of the multi-dimensional rules:
enum Rank { R_NONE, R_LIN, R_QUAD, R_CUBIC };

template <int N, bool IN>
__device__ __forceinline__ Rank rank_of(int j, int last) {
    const bool has2 = IN || last >= j + 1, has3 = j + 2 <= N && (IN || last >= j + 2);
    if (!has2) return R_NONE;
    return j == 0 ? (has3 ? R_QUAD : R_LIN) : (has3 ? R_CUBIC : R_QUAD);
}

// The value of the formula of point j's rank; v0..v3 are the known values
// j - 1 .. j + 2 (anything where there is none).  R_NONE keeps v1.
template <typename T, int N, bool IN>
__device__ __forceinline__ T pred_line(int j, int last, T v0, T v1, T v2, T v3) {
    if constexpr (IN) {
        if (N == 1) return lin(v1, v2);
        return j == 0 ? quad_r(v1, v2, v3) : (j == N - 1 ? quad_l(v0, v1, v2) : cubic(v0, v1, v2, v3));
    } else {
        T p = v1;
        if (last >= j + 1) p = j == 0 ? lin(v1, v2) : quad_l(v0, v1, v2);
        if (j + 2 <= N && last >= j + 2) p = j == 0 ? quad_r(v1, v2, v3) : cubic(v0, v1, v2, v3);
        return p;
    }
}

// ------------------------------------------------------------------ stages --
// Where a compressing stage puts its codes: straight to the level-major
// array (levels 1-3), into registers (the first two stages of level 0, whose
// values later stages still read), or into the points' own slots (the last
// stage of level 0).  Level 0's codes then leave the tile as whole rows.
enum Sink { TO_GLOBAL, TO_REGS, TO_SLOT };
struct RegCodes {
    int32_t code[8];
    int slot, step;  // slot of code 0 (-1: none to store), distance of the slots
};

// Level-major index step from point j of a line along A to point j + 1 (the
// coordinate keeps its parity); y, z: the line's fixed coordinates.
template <int L, int A, typename T, bool IN>
__device__ __forceinline__ uint32_t lm_step(const Tile<T, IN>& t, int y, int z) {
    if constexpr (A == 0) return (((y | z) >> L) & 1) ? 2u : 1u;
    if constexpr (A == 1)
        return 2u * (uint32_t)t.g.lx[L] - (((z >> L) & 1) ? 0u : (uint32_t)t.g.lx[L + 1]);
    return 2u * (uint32_t)t.g.lxy[L] - (uint32_t)t.g.lxy[L + 1];
}

template <int L, typename T, bool IN>
__device__ __forceinline__ uint32_t lm_at(const Tile<T, IN>& t, int x, int y, int z) {
    return lm_index<L>(t.g, t.ox + x, t.oy + y, t.oz + z);
}

template <int U>
constexpr int level_of_unit() {
    return U == 1 ? 0 : (U == 2 ? 1 : (U == 4 ? 2 : 3));
}

// One point: its slot's value (or code) against pred.
template <typename T, int M, int SINK, bool IN>
__device__ __forceinline__ void put_point(Tile<T, IN>& t, int slot, T v, T pred, int32_t& code) {
    if constexpr (M == COMPRESS) {
        code = quantize_val(v, pred, t.eb_r, t.ebx2);
        t.s[slot] = SINK == TO_SLOT ? code_slot(code, T()) : v;
    } else {
        t.s[slot] = pred + (T)slot_code(v) * t.ebx2;
    }
}

// The N points of one line per lane: known values at slots base + j * step,
// points at base + half + j * step (step and half: compile-time constants,
// or per-lane values where the lanes' lines differ in direction).
template <typename T, int U, int M, int SINK, bool IN, class Step, class Half>
__device__ __forceinline__ void line_points(Tile<T, IN>& t, int base, Step step, Half half, int r, bool own,
                                            uint32_t idx, uint32_t idx_step, RegCodes* rc) {
    constexpr int N = 8 / U;
    const int last = (int)((unsigned)(r - 1) / (2 * U));
    T k[N + 1], v[N];
#pragma unroll
    for (int j = 0; j <= N; ++j) k[j] = t.s[base + j * step];
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = t.s[base + half + j * step];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const T pred = pred_line<T, N, IN>(j, last, k[j > 0 ? j - 1 : 0], k[j], k[j + 1], k[j + 2 <= N ? j + 2 : N]);
        int32_t code;
        put_point<T, M, SINK>(t, base + half + j * step, v[j], pred, code);
        if constexpr (M == COMPRESS && SINK == TO_GLOBAL) {
            if (own && (IN || (2 * j + 1) * U < r)) t.qc_out[idx + j * idx_step] = code;
        }
        if constexpr (M == COMPRESS && SINK == TO_REGS) rc->code[j] = code;
    }
    if constexpr (M == COMPRESS && SINK == TO_REGS) {
        rc->slot = own ? base + half : -1;
        rc->step = step;
    }
}

// A 1-D stage: lines along A over the other two axes, P (the lower) fastest;
// ALLP / ALLQ: at every multiple of U, or at the even ones.  EXCL: the last
// stage of level 0, own points only (x, y, z < 16).
template <typename T, int U, int A, bool ALLP, bool ALLQ, bool EXCL, int M, int SINK, bool IN>
__device__ __forceinline__ void line_stage(Tile<T, IN>& t, RegCodes* rc = nullptr) {
    constexpr int N = 8 / U, L = level_of_unit<U>();
    constexpr int CP = EXCL ? 16 : (ALLP ? 2 * N + 1 : N + 1), CQ = EXCL ? 16 : (ALLQ ? 2 * N + 1 : N + 1);
    static_assert(CP * CQ <= kThreads, "one line per lane");
    if constexpr (M == COMPRESS && SINK == TO_REGS) rc->slot = -1;
    const int l = lane_id();
    if (l < CP * CQ) {
        const int p = (l % CP) * (ALLP ? U : 2 * U), q = (l / CP) * (ALLQ ? U : 2 * U);
        const int x = A == 0 ? 0 : p, y = A == 1 ? 0 : (A == 0 ? p : q), z = A == 2 ? 0 : q;
        if (t.template in<A == 0 ? 1 : 0>(p) && t.template in<A == 2 ? 1 : 2>(q)) {
            const bool own = p < 16 && q < 16;
            uint32_t idx = 0, idx_step = 0;
            if constexpr (M == COMPRESS && SINK == TO_GLOBAL) {
                idx = lm_at<L>(t, A == 0 ? U : x, A == 1 ? U : y, A == 2 ? U : z);
                idx_step = lm_step<L, A>(t, y, z);
            }
            line_points<T, U, M, SINK>(t, tslot(x, y, z), std::integral_constant<int, slot_step<U, A>()>{},
                                       std::integral_constant<int, slot_half<U, A>()>{},
                                       A == 0 ? t.rx : (A == 1 ? t.ry : t.rz), own, idx, idx_step, rc);
        }
    }
    lds_barrier();
}

// LINE points (one odd coordinate): the lines along x, y and z through the
// points with both other coordinates even, in one sweep.
template <typename T, int U, int M, int SINK, bool IN>
__device__ __forceinline__ void lines3_stage(Tile<T, IN>& t, RegCodes* rc = nullptr) {
    constexpr int N = 8 / U, C = N + 1, L = level_of_unit<U>();
    static_assert(3 * C * C <= kThreads, "one line per lane");
    if constexpr (M == COMPRESS && SINK == TO_REGS) rc->slot = -1;
    const int l = lane_id();
    if (l < 3 * C * C) {
        const int grp = l / (C * C), m = l % (C * C), i = 2 * U * (m % C), j = 2 * U * (m / C);
        const int x = grp == 0 ? 0 : i, y = grp == 0 ? i : (grp == 1 ? 0 : j), z = grp == 2 ? 0 : j;
        if (t.in3(x, y, z)) {
            const int step = grp == 0 ? slot_step<U, 0>() : (grp == 1 ? slot_step<U, 1>() : slot_step<U, 2>());
            const int half = grp == 0 ? slot_half<U, 0>() : (grp == 1 ? slot_half<U, 1>() : slot_half<U, 2>());
            const int r = grp == 0 ? t.rx : (grp == 1 ? t.ry : t.rz);
            uint32_t idx = 0, idx_step = 0;
            if constexpr (M == COMPRESS && SINK == TO_GLOBAL) {
                idx = lm_at<L>(t, grp == 0 ? U : x, grp == 1 ? U : y, grp == 2 ? U : z);
                idx_step = grp == 0 ? lm_step<L, 0>(t, 0, 0) : (grp == 1 ? lm_step<L, 1>(t, 0, 0) : lm_step<L, 2>(t, 0, 0));
            }
            line_points<T, U, M, SINK>(t, tslot(x, y, z), step, half, r, i < 16 && j < 16, idx, idx_step, rc);
        }
    }
    lds_barrier();
}

// FACE points (two odd coordinates, InterpolationPredictor.cu:1546-1669): a
// lane takes a line of N points along A (z, or y for the points with even
// z) at one odd position jb of the other odd axis B.  The two directions'
// formulas compete by rank: equal ranks are averaged, the higher one wins,
// and where neither has a far neighbour the point continues the plane
// through its three known neighbours.
template <typename T, int U, int M, int SINK, bool IN>
__device__ __forceinline__ void faces_stage(Tile<T, IN>& t, RegCodes* rc = nullptr) {
    constexpr int N = 8 / U, C = N + 1, L = level_of_unit<U>();
    static_assert(3 * N * C <= kThreads, "one line per lane");
    if constexpr (M == COMPRESS && SINK == TO_REGS) rc->slot = -1;
    const int l = lane_id();
    if (l < 3 * N * C) {
        // groups: (y, z) odd at even x; (x, z) odd at even y; (x, y) odd at even z
        const int grp = l / (N * C), m = l % (N * C);
        const int jb = grp == 1 ? m % N : m / C, ic = grp == 1 ? m / N : m % C;
        const int c = 2 * U * ic, b = 2 * U * jb;  // even axis; left neighbour along B
        const int x = grp == 0 ? c : b, y = grp == 0 ? b : (grp == 1 ? c : 0), z = grp == 2 ? c : 0;
        if (t.in3(grp == 0 ? x : x + U, grp == 1 ? y : y + U, grp == 2 ? z : z + U)) {
            const int sa = grp == 2 ? slot_step<U, 1>() : slot_step<U, 2>();
            const int ha = grp == 2 ? slot_half<U, 1>() : slot_half<U, 2>();
            const int sb = grp == 0 ? slot_step<U, 1>() : slot_step<U, 0>();
            const int hb = grp == 0 ? slot_half<U, 1>() : slot_half<U, 0>();
            const int left = tslot(x, y, z);  // A and B even
            const int ka = left + hb;         // A even, B odd: known values along A
            const int own_slot = ka + ha;     // the points
            const int p1 = left + ha, p0 = p1 - (jb > 0 ? sb : 0), p2 = p1 + sb, p3 = p2 + (jb < N - 1 ? sb : 0);
            const int ra = grp == 2 ? t.ry : t.rz, rb = grp == 0 ? t.ry : t.rx;
            const int lasta = (int)((unsigned)(ra - 1) / (2 * U)), lastb = (int)((unsigned)(rb - 1) / (2 * U));
            const bool own = c < 16;
            uint32_t idx = 0, idx_step = 0;
            if constexpr (M == COMPRESS && SINK == TO_GLOBAL) {
                idx = lm_at<L>(t, grp == 0 ? x : x + U, grp == 1 ? y : y + U, grp == 2 ? z : z + U);
                idx_step = grp == 2 ? lm_step<L, 1>(t, 0, 0) : lm_step<L, 2>(t, 0, 0);
            }
            const bool b3 = jb > 0 && jb + 2 <= N && (IN || lastb >= jb + 2);  // B's formula is the cubic
            T k[N + 1];
#pragma unroll
            for (int j = 0; j <= N; ++j) k[j] = t.s[ka + j * sa];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int o = j * sa;
                const T v0 = t.s[p0 + o], v1 = t.s[p1 + o], v2 = t.s[p2 + o], v3 = t.s[p3 + o];
                const T a0 = k[j > 0 ? j - 1 : 0], a1 = k[j], a2 = k[j + 1], a3 = k[j + 2 <= N ? j + 2 : N];
                T pred;
                if constexpr (IN) {
                    const T pa = pred_line<T, N, true>(j, N, a0, a1, a2, a3);
                    if (N == 1) {
                        pred = (pa + lin(v1, v2)) / (T)2;
                    } else if (j == 0 || j == N - 1) {
                        const T qb = jb == 0 ? quad_r(v1, v2, v3) : quad_l(v0, v1, v2);
                        pred = (pa + qb) / (T)2;
                        if (N > 2) pred = b3 ? cubic(v0, v1, v2, v3) : pred;
                    } else {
                        const T both = (pa + cubic(v0, v1, v2, v3)) / (T)2;
                        pred = b3 ? both : pa;
                    }
                } else {
                    const Rank fa = rank_of<N, false>(j, lasta), fb = rank_of<N, false>(jb, lastb);
                    const T pa = pred_line<T, N, false>(j, lasta, a0, a1, a2, a3);
                    T pb = fb == R_CUBIC ? cubic(v0, v1, v2, v3) : quad_l(v0, v1, v2);
                    if (jb == 0) pb = fb == R_QUAD ? quad_r(v1, v2, v3) : lin(v1, v2);
                    pred = fa > fb ? pa : pb;
                    if (fa == fb) {
                        if (fa == R_NONE) pred = (a1 + v1) - t.s[left + o];
                        else pred = (pa + pb) / (T)2;
                    }
                }
                int32_t code;
                put_point<T, M, SINK>(t, own_slot + o, t.s[own_slot + o], pred, code);
                if constexpr (M == COMPRESS && SINK == TO_GLOBAL) {
                    if (own && (IN || (2 * j + 1) * U < ra)) t.qc_out[idx + j * idx_step] = code;
                }
                if constexpr (M == COMPRESS && SINK == TO_REGS) rc->code[j] = code;
            }
            if constexpr (M == COMPRESS && SINK == TO_REGS) {
                rc->slot = own ? own_slot : -1;
                rc->step = sa;
            }
        }
    }
    lds_barrier();
}

// CUBE points (three odd coordinates, InterpolationPredictor.cu:1671-1723):
// the mean of the directions whose formula is the cubic; without one, x's
// formula.
template <typename T, int U, int M, int SINK, bool IN>
__device__ __forceinline__ void cubes_stage(Tile<T, IN>& t) {
    constexpr int N = 8 / U, L = level_of_unit<U>(), TOTAL = N * N * N;
    constexpr int SX = slot_step<U, 0>(), SY = slot_step<U, 1>(), SZ = slot_step<U, 2>();
    constexpr int HX = slot_half<U, 0>(), HY = slot_half<U, 1>(), HZ = slot_half<U, 2>();
    const int l = lane_id();
#pragma unroll
    for (int it = 0; it < (TOTAL + kThreads - 1) / kThreads; ++it) {
        const int p = l + it * kThreads;
        if (TOTAL % kThreads == 0 || p < TOTAL) {
            const int i = p % N, j = (p / N) % N, k = p / (N * N);
            const int x = (2 * i + 1) * U, y = (2 * j + 1) * U, z = (2 * k + 1) * U;
            if (t.in3(x, y, z)) {
                const int lastx = (int)((unsigned)(t.rx - 1) / (2 * U)), lasty = (int)((unsigned)(t.ry - 1) / (2 * U)),
                          lastz = (int)((unsigned)(t.rz - 1) / (2 * U));
                const int corner = i * SX + j * SY + k * SZ, own_slot = corner + HX + HY + HZ;
                // x's taps: y and z odd, from the left neighbour
                const int bx = corner + HY + HZ;
                const T x0 = t.s[bx - (i > 0 ? SX : 0)], x1 = t.s[bx], x2 = t.s[bx + SX];
                const T x3 = t.s[bx + (i < N - 1 ? 2 * SX : SX)];
                const Rank fx = rank_of<N, IN>(i, lastx);
                T pred = x1;
                if (N > 1 && fx == R_QUAD) pred = i == 0 ? quad_r(x1, x2, x3) : quad_l(x0, x1, x2);
                if ((N == 1 || !IN) && fx == R_LIN) pred = lin(x1, x2);
                if constexpr (N > 2) {
                    const int by = corner + HX + HZ, bz = corner + HX + HY;
                    const int y0 = by - (j > 0 ? SY : 0), y3 = by + (j < N - 1 ? 2 * SY : SY);
                    const int z0 = bz - (k > 0 ? SZ : 0), z3 = bz + (k < N - 1 ? 2 * SZ : SZ);
                    const T px = cubic(x0, x1, x2, x3);
                    const T py = cubic(t.s[y0], t.s[by], t.s[by + SY], t.s[y3]);
                    const T pz = cubic(t.s[z0], t.s[bz], t.s[bz + SZ], t.s[z3]);
                    const bool cx = fx == R_CUBIC, cy = rank_of<N, IN>(j, lasty) == R_CUBIC,
                               cz = rank_of<N, IN>(k, lastz) == R_CUBIC;
                    // an absent direction adds 0 (a zero's sign cannot reach a
                    // value or code: each adds code * ebx2 to the prediction)
                    const T sum = ((cx ? px : (T)0) + (cy ? py : (T)0)) + (cz ? pz : (T)0);
                    const int n = (int)cx + (int)cy + (int)cz;
                    if (n == 1) pred = sum;
                    if (n == 2) pred = sum / (T)2;
                    if (n == 3) pred = sum / (T)3;
                }
                int32_t code;
                put_point<T, M, SINK>(t, own_slot, t.s[own_slot], pred, code);
                if constexpr (M == COMPRESS && SINK == TO_GLOBAL) t.qc_out[lm_at<L>(t, x, y, z)] = code;
            }
        }
    }
    lds_barrier();
}

// Level 0's codes of the 16^3 tile, in their slots once the register-held
// ones join them, written out row by row: lane (x, y) = (l mod 16, l / 16)
// takes z = 0..15.  A row (y, z) with y or z odd holds every x (16 adjacent
// codes), the others the odd x (8 adjacent codes); from z to z + 2 the index
// advances by 2 lxy0 - lxy1.
template <typename T, bool IN>
__device__ __forceinline__ void level0_codes_out(Tile<T, IN>& t, const RegCodes& a, const RegCodes& b) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (a.slot >= 0) t.s[a.slot + k * a.step] = code_slot(a.code[k], T());
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (b.slot >= 0) t.s[b.slot + k * b.step] = code_slot(b.code[k], T());
    }
    lds_barrier();
    const int lane = lane_id();
    const int x = lane & 15, y = lane >> 4;
    if (!(t.template in<0>(x) && t.template in<1>(y))) return;
    const int64_t step = 2 * t.g.lxy[0] - t.g.lxy[1];
    const T* src = t.s + tslot(x, y, 0);
    int32_t* odd = t.qc_out + lm_at<0>(t, x, y, 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (t.template in<2>(2 * k + 1)) *odd = slot_code(src[(2 * k + 1) * kZP]);
        odd += step;
    }
    if ((x | y) & 1) {
        int32_t* even = t.qc_out + lm_at<0>(t, x, y, 0);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (t.template in<2>(2 * k)) *even = slot_code(src[2 * k * kZP]);
            even += step;
        }
    }
}

// The three stages of one level (InterpolationPredictor.cu:1940-2025).
template <typename T, int U, int M, bool IN>
__device__ __forceinline__ void level3(Tile<T, IN>& t, bool md, bool rev) {
    constexpr bool EX = U == 1;
    constexpr int S1 = U == 1 ? TO_REGS : TO_GLOBAL, S2 = U == 1 ? TO_SLOT : TO_GLOBAL;
    RegCodes a, b;
    if (md) {
        lines3_stage<T, U, M, S1>(t, &a);
        faces_stage<T, U, M, S1>(t, &b);
        cubes_stage<T, U, M, S2>(t);
    } else if (rev) {
        line_stage<T, U, 0, false, false, false, M, S1>(t, &a);
        line_stage<T, U, 1, true, false, false, M, S1>(t, &b);
        line_stage<T, U, 2, true, true, EX, M, S2>(t);
    } else {
        line_stage<T, U, 2, false, false, false, M, S1>(t, &a);
        line_stage<T, U, 1, false, true, false, M, S1>(t, &b);
        line_stage<T, U, 0, true, true, EX, M, S2>(t);
    }
    if constexpr (M == COMPRESS && U == 1) level0_codes_out(t, a, b);
}

// The four levels of a tile, coarsest first.
template <typename T, int M, bool IN>
__device__ __forceinline__ void tile_levels(Tile<T, IN>& t, const LevelEb<T>& le, const uint8_t* flags8, int maxlevel) {
    uint8_t fl[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) fl[i] = flags8[i];
    if (3 <= maxlevel) { t.eb_r = le.eb_r[3]; t.ebx2 = le.ebx2[3]; level3<T, 8, M>(t, fl[3], fl[7]); }
    if (2 <= maxlevel) { t.eb_r = le.eb_r[2]; t.ebx2 = le.ebx2[2]; level3<T, 4, M>(t, fl[2], fl[6]); }
    if (1 <= maxlevel) { t.eb_r = le.eb_r[1]; t.ebx2 = le.ebx2[1]; level3<T, 2, M>(t, fl[1], fl[5]); }
    if (0 <= maxlevel) { t.eb_r = le.eb_r[0]; t.ebx2 = le.ebx2[0]; level3<T, 1, M>(t, fl[0], fl[4]); }
}

// ------------------------------------------------------- tile and memory --
// The 17^3 points of a tile are taken as 20 sets of at most one point per
// lane: the column (x, y) = (l mod 16, l / 16) at z = 0..16, then the faces
// y = 16 (lane (x, z)) and x = 16 (lane (y, z)) without their last rows, then
// those rows: (x, 16, 16), (16, 16, z) and (16, y, 16).  Addresses advance by
// one plane from point to point, so a column costs one addition per point.
// false: the lane has no point.
__device__ __forceinline__ bool edge_point(int l, int& x, int& y, int& z) {
    x = l < 16 ? l : 16;
    y = l < 33 ? 16 : l - 33;
    z = l >= 16 && l < 33 ? l - 16 : 16;
    return l < 49;
}

// Tile plus halo into LDS: all global loads of a lane are issued before the
// first LDS write so the tile costs one memory latency.  Points outside the
// field are not read (no formula uses their slots).
template <typename T, bool IN>
__device__ __forceinline__ void tile_load(const Tile<T, IN>& t, const T* __restrict__ data) {
    const int l = lane_id();
    const int x = l & 15, y = l >> 4;
    const int64_t nx = t.g.nx, nxy = nx * t.g.ny;
    const T* base = data + (t.oz * nxy + t.oy * nx + t.ox);
    T v[17], fy = (T)0, fx = (T)0, e = (T)0;
    int ex, ey, ez;
    const bool edge = edge_point(l, ex, ey, ez);
    const bool on = t.template in<0>(x) && t.template in<1>(y);
    const T* p = base + (y * nx + x);
#pragma unroll
    for (int z = 0; z < 17; ++z) {
        v[z] = (T)0;
        if (on && t.template in<2>(z)) v[z] = *p;
        p += nxy;
    }
    if (t.in3(x, 16, y)) fy = base[y * nxy + 16 * nx + x];
    if (t.in3(16, x, y)) fx = base[y * nxy + x * nx + 16];
    if (edge && t.in3(ex, ey, ez)) e = base[ez * nxy + ey * nx + ex];
    T* d = t.s + tslot(x, y, 0);
#pragma unroll
    for (int z = 0; z < 17; ++z) d[z * kZP] = v[z];
    t.s[tslot(x, 16, y)] = fy;
    t.s[tslot(16, x, y)] = fx;
    if (edge) t.s[tslot(ex, ey, ez)] = e;
}

// Decompression first fills the slot of every point with the bit pattern of
// its own code (corners: the anchors; points of skipped levels: 0); a stage
// then reads the slot of the point it reconstructs and overwrites it.  E:
// int32_t or int16_t codes.
template <typename T>
struct TileCodes {
    int32_t v0[17], fy, fx, e;  // level 0, the point sets above
    int32_t v1[3], v23;         // levels 1 (9^3 points), 2 (5^3, lanes 0..) and 3 (3^3, lanes 128..)
    T anc;
};

// the tile's eight corner anchors (x_reset_scratch_data 1051-1061)
template <typename T, bool IN>
__device__ __forceinline__ T anchor_load(const Tile<T, IN>& t, const T* __restrict__ anchors, int bx, int by, int bz) {
    const int l = lane_id();
    T a = (T)0;
    if (l < 8) {
        const int ax = bx + (l & 1), ay = by + ((l >> 1) & 1), az = bz + (l >> 2);
        if (anchors && ax < t.g.gx && ay < t.g.gy && az < t.g.gz)
            a = anchors[ax + (int64_t)ay * t.g.gx + (int64_t)az * t.g.gx * t.g.gy];
    }
    return a;
}

template <typename T, bool IN>
__device__ __forceinline__ void anchor_store(const Tile<T, IN>& t, T anc) {
    const int l = lane_id();
    if (l < 8) t.s[tslot(16 * (l & 1), 16 * ((l >> 1) & 1), 16 * (l >> 2))] = anc;
}

// lane's point of levels 2 and 3 in lattice units
__device__ __forceinline__ bool coarse_point(int l, int& unit, int& i, int& j, int& k) {
    const bool l3 = l >= 128;
    const int m = l3 ? l - 128 : l;
    unit = l3 ? 8 : 4;
    i = l3 ? m % 3 : m % 5;
    j = l3 ? (m / 3) % 3 : (m / 5) % 5;
    k = l3 ? m / 9 : m / 25;
    return m < (l3 ? 27 : 125);
}

template <typename T, bool IN, typename E>
__device__ __forceinline__ void codes_load(const Tile<T, IN>& t, const E* __restrict__ q, int maxlevel,
                                           const T* __restrict__ anchors, int bx, int by, int bz, TileCodes<T>& c) {
    const int l = lane_id();
    const int x = l & 15, y = l >> 4;
    const bool l0 = maxlevel >= 0;
    c.v23 = 0;
    {
        int u, i, j, k;
        if (coarse_point(l, u, i, j, k) && ((i | j | k) & 1) && t.in3(u * i, u * j, u * k)) {
            if (u == 4) {
                if (maxlevel >= 2) c.v23 = q[lm_at<2>(t, 4 * i, 4 * j, 4 * k)];
            } else if (maxlevel >= 3) {
                c.v23 = q[lm_at<3>(t, 8 * i, 8 * j, 8 * k)];
            }
        }
    }
#pragma unroll
    for (int it = 0; it < 3; ++it) {
        const int p = l + it * kThreads, i = p % 9, j = (p / 9) % 9, k = p / 81;
        c.v1[it] = 0;
        if (maxlevel >= 1 && p < 729 && ((i | j | k) & 1) && t.in3(2 * i, 2 * j, 2 * k))
            c.v1[it] = q[lm_at<1>(t, 2 * i, 2 * j, 2 * k)];
    }
    const int64_t step = 2 * t.g.lxy[0] - t.g.lxy[1];
    const bool on = l0 && t.template in<0>(x) && t.template in<1>(y), on_even = on && ((x | y) & 1);
    const E* even = q + lm_at<0>(t, x, y, 0);
    const E* odd = q + lm_at<0>(t, x, y, 1);
#pragma unroll
    for (int k = 0; k <= 8; ++k) {
        c.v0[2 * k] = 0;
        if (on_even && t.template in<2>(2 * k)) c.v0[2 * k] = *even;
        even += step;
        if (k < 8) {
            c.v0[2 * k + 1] = 0;
            if (on && t.template in<2>(2 * k + 1)) c.v0[2 * k + 1] = *odd;
            odd += step;
        }
    }
    c.fy = c.fx = c.e = 0;
    if (l0 && ((x | y) & 1)) {  // z = y here, then y = x
        if (t.in3(x, 16, y)) c.fy = q[lm_at<0>(t, x, 16, y)];
        if (t.in3(16, x, y)) c.fx = q[lm_at<0>(t, 16, x, y)];
    }
    int ex, ey, ez;
    if (edge_point(l, ex, ey, ez) && l0 && ((ex | ey | ez) & 1) && t.in3(ex, ey, ez)) c.e = q[lm_at<0>(t, ex, ey, ez)];
    c.anc = anchor_load(t, anchors, bx, by, bz);
}

template <typename T, bool IN>
__device__ __forceinline__ void codes_store(const Tile<T, IN>& t, const TileCodes<T>& c) {
    const int l = lane_id();
    const int x = l & 15, y = l >> 4;
    {
        int u, i, j, k;
        if (coarse_point(l, u, i, j, k) && ((i | j | k) & 1)) t.s[tslot(u * i, u * j, u * k)] = code_slot(c.v23, T());
    }
#pragma unroll
    for (int it = 0; it < 3; ++it) {
        const int p = l + it * kThreads, i = p % 9, j = (p / 9) % 9, k = p / 81;
        if (p < 729 && ((i | j | k) & 1)) t.s[tslot(2 * i, 2 * j, 2 * k)] = code_slot(c.v1[it], T());
    }
    T* d = t.s + tslot(x, y, 0);
#pragma unroll
    for (int k = 0; k < 8; ++k) d[(2 * k + 1) * kZP] = code_slot(c.v0[2 * k + 1], T());
    if ((x | y) & 1) {
#pragma unroll
        for (int k = 0; k <= 8; ++k) d[2 * k * kZP] = code_slot(c.v0[2 * k], T());
        t.s[tslot(x, 16, y)] = code_slot(c.fy, T());
        t.s[tslot(16, x, y)] = code_slot(c.fx, T());
    }
    int ex, ey, ez;
    if (edge_point(l, ex, ey, ez) && ((ex | ey | ez) & 1)) t.s[tslot(ex, ey, ez)] = code_slot(c.e, T());
    anchor_store(t, c.anc);
}

}  // namespace
}  // namespace pa
