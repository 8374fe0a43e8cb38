// resident.hip -- the kernels of resident.hpp.
#include "resident.hpp"

#include <algorithm>
#include <type_traits>

#include "engine_strip.hpp"

namespace tea {
namespace res {
namespace {

// 100 MHz counter: how long to wait for the other workgroups to start, and
// for an exchange once all have.
constexpr long long START_TICKS = 20000000;       // 0.2 s
constexpr long long EXCHANGE_TICKS = 1000000000;  // 10 s
// How long a wave waits (64 clocks each) before its first look for the other
// workgroups' sums where it has nothing else to do meanwhile, and between two
// looks: 255 workgroups reading the same lines hold up the stores they wait
// for (a CG deck of 1000^2 cells, 879 iterations: 7.6 ms; without the first wait
// 8.7, with one copy of the sums instead of eight 8.4, without both 9.9).
constexpr int FIRST_LOOK = 24, NEXT_LOOK = 2;

__device__ __forceinline__ word_t load_word(const word_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_word(word_t *p, unsigned tag, unsigned data)
{
    __hip_atomic_store(p, ((word_t)tag << 32) | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// The rows of a wave with `mine` strips sit in v[0 .. 4 mine); v[4 mine] holds
// the row above them.  set_top, get_top, get_last: that row and the one below
// it for a run-time count, by selects among registers (the empty asm keeps the
// compiler from making the array an indexed one, which would move it out of
// the registers).
template <int S, typename T, int N> __device__ __forceinline__ void set_top(T (&v)[N], int mine, T t)
{
#pragma unroll
    for (int k = 1; k <= S; k++) {
        T a = v[k * STRIP];
        asm("" : "+v"(a));
        v[k * STRIP] = k == mine ? t : a;
    }
}
template <int S, int BACK, typename T, int N> __device__ __forceinline__ T get_row(const T (&v)[N], int mine)
{
    T t = v[STRIP - BACK];
#pragma unroll
    for (int k = 2; k <= S; k++) {
        T a = v[k * STRIP - BACK];
        asm("" : "+v"(a));
        t = k == mine ? a : t;
    }
    return t;
}
template <int S, typename T, int N> __device__ __forceinline__ T get_top(const T (&v)[N], int mine)
{
    return get_row<S, 0>(v, mine);
}
template <int S, typename T, int N> __device__ __forceinline__ T get_last(const T (&v)[N], int mine)
{
    return get_row<S, 1>(v, mine);
}

// What a workgroup shares in LDS besides the preconditioner's factors.
template <typename T, int S> struct Shared {
    static constexpr int R = S * STRIP;
    static constexpr int NW = R * (int)sizeof(T) / 4;   // 32-bit words of a column face per wave
    static_assert(NW <= FACE_WORDS, "a lane per word");
    unsigned face[RES_WAVES][2][NW];    // column faces on their way out and in
    T rows[2][RES_WAVES][2][WAVE];      // [slot] first and last row of each wave
    DD part[2][RES_WAVES];
    DD sum[2][RES_MAX_WG / WAVE];       // all-reduced: one sum per 64 workgroups
    int verdict, bad;
};

__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wave's place in the tiles, and the exchanges it takes part in.
template <typename T, int S> struct Place {
    static constexpr int R = S * STRIP;
    using Sh = Shared<T, S>;
    int lane, wave, wg, nbx, nwg;
    int c, r0, nrows;       // column; first row and rows of this wave
    int mine;               // its strips
    int nout;               // columns of the band (lanes 1 .. nout)
    int lastw;              // the tile's last wave with rows
    bool out, col_in, col_mem;
    bool left, right, below, above;   // neighbouring tiles
    bool in_below, in_above;          // the rows below and above the wave are inside the mesh
    long pitch;
    unsigned row_b, bytes;            // bytes per row and in all of a field
    unsigned o_out, o_in, o_mem;      // this lane's column in row r0 for lanes that own it, lie in the mesh, exist; else OOB
    Exchange x;
    unsigned rtag, xtag;    // tags of the latest reduction and exchange

    __device__ Place(const Tiles &t, const Exchange &ex) : pitch(t.pitch), x(ex)
    {
        lane = threadIdx.x & (WAVE - 1);
        wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
        wg = blockIdx.x;
        nbx = t.nbx;
        nwg = t.nbx * t.nby;
        const int bx = wg % t.nbx, by = wg / t.nbx;
        const int ny = t.e.y1 - t.e.y0 + 1, nstrips = (ny + STRIP - 1) / STRIP;
        const int cfirst = t.e.x0 + bx * t.ow;
        nout = min(t.ow, t.e.x1 - cfirst + 1);
        c = cfirst - 1 + lane;
        col_mem = lane <= nout + 1;
        col_in = col_mem && c >= t.e.x0 && c <= t.e.x1;
        out = lane >= 1 && lane <= nout;
        const int ts = min(t.ts, nstrips - by * t.ts);        // strips of this tile
        const int each = ts / RES_WAVES, extra = ts % RES_WAVES;
        mine = each + (wave < extra ? 1 : 0);
        r0 = t.e.y0 + (by * t.ts + wave * each + min(wave, extra)) * STRIP;
        nrows = max(0, min(mine * STRIP, t.e.y1 - r0 + 1));
        lastw = min(ts, RES_WAVES) - 1;
        left = bx > 0;
        right = bx < t.nbx - 1;
        below = by > 0;
        above = by < t.nby - 1;
        in_below = r0 - 1 >= t.e.y0;
        in_above = r0 + nrows <= t.e.y1;
        row_b = (unsigned)(pitch * sizeof(T));
        bytes = (unsigned)(t.e.y1 + 2) * row_b;
        const unsigned o = (unsigned)r0 * row_b + (unsigned)(c * (int)sizeof(T));
        o_out = out ? o : OOB;
        o_in = col_in ? o : OOB;
        o_mem = col_mem ? o : OOB;
        rtag = xtag = ex.tag;
    }

    __device__ int strip_len(int k) const { return max(0, min(STRIP, nrows - k * STRIP)); }
    // Sets what strip k has beyond its rows to 0 (a test per strip: only a
    // tile's last one, at the top of the mesh, is ever short).
    template <int N> __device__ void cut(int k, T (&v)[N], int at = 0) const
    {
        if ((k + 1) * STRIP <= nrows) return;
        asm volatile("" ::: "memory");   // a branch, not selects on every row
#pragma unroll
        for (int i = 0; i < STRIP; i++)
            if (k * STRIP + i >= nrows) v[at + i] = T(0.0);
    }
    // acc without the lanes that own no column
    __device__ DD owned(DD acc) const { return DD{out ? acc.s : 0.0, out ? acc.c : 0.0}; }
    // row r0 + j (j < n) at lane offset o
    __device__ T load(const FieldBuf<T> &b, unsigned o, int j, int n) const
    {
        return b.load(j < n ? o : OOB, (unsigned)j * row_b);
    }
    __device__ void store(const FieldBuf<T> &b, unsigned o, int j, int n, T v) const
    {
        b.store(j < n ? o : OOB, v, (unsigned)j * row_b);
    }
    // the row below r0
    __device__ T load_below(const FieldBuf<T> &b, unsigned o) const
    {
        return b.load(nrows > 0 && o != OOB ? o - row_b : OOB);
    }
    __device__ FieldBuf<T> field(const T *f) const { return FieldBuf<T>(f, bytes); }

    // Post this wave's values of the exchanged field: the column faces
    // (through LDS, so that one store instruction carries both), the rows
    // shared with the waves below and above (LDS), and the tile's outer rows.
    template <int N> __device__ void post(Sh &sh, const T (&v)[N])
    {
        xtag++;
        const int slot = xtag & 1;
        if (nrows == 0) return;
        const T last = get_last<S>(v, mine);   // (a strip cut short has no row above it)
        sh.rows[slot][wave][0][lane] = v[0];
        sh.rows[slot][wave][1][lane] = last;
        if (below && wave == 0) post_row(slot, 0, v[0]);
        if (above && wave == lastw) post_row(slot, 1, last);
        if (left || right) {
            unsigned *f = &sh.face[wave][lane == 1 ? 0 : 1][0];
            if (lane == 1 || lane == nout) {
#pragma unroll
                for (int j = 0; j < R; j++) put(f, j, v[j]);
            }
            wave_lds_fence();
            const bool mine_too = lane < nrows * (int)sizeof(T) / 4;
            if (left && mine_too) store_word(col_at(slot, wg, 0), xtag, sh.face[wave][0][lane]);
            if (right && mine_too) store_word(col_at(slot, wg, 1), xtag, sh.face[wave][1][lane]);
            wave_lds_fence();
        }
    }

    // What the neighbours posted under the current tag: column values into v
    // of the halo lanes (0 and nout + 1), the rows just below and above the
    // wave into vb and vt.  Follows a barrier (the rows of the tile's other
    // waves).  Lanes and rows without a neighbour keep their values.
    template <int N> __device__ void take(Sh &sh, T (&v)[N], T &vb, T &vt)
    {
        if (nrows == 0) return;
        const int slot = xtag & 1;
        if (wave > 0) vb = sh.rows[slot][wave - 1][1][lane];
        if (wave < lastw) vt = sh.rows[slot][wave + 1][0][lane];
        const bool wc = lane < nrows * (int)sizeof(T) / 4, wl = wc && left, wr = wc && right;
        // the left neighbour's right face, the right neighbour's left face
        const word_t *pl = col_at(slot, wg - 1, 1), *pr = col_at(slot, wg + 1, 0);
        const bool wb = below && wave == 0 && out, wt = above && wave == lastw && out;
        const word_t *pb = row_at(slot, wg - nbx, 1), *pt = row_at(slot, wg + nbx, 0);
        word_t ql = 0, qr = 0;
        T nb = T(0.0), nt = T(0.0);
        if (!poll(sh, [&] {
                bool ok = true;
                if (wl) ql = load_word(pl);
                if (wr) qr = load_word(pr);
                if (wl) ok = (unsigned)(ql >> 32) == xtag;
                if (wr) ok = ok && (unsigned)(qr >> 32) == xtag;
                if (wb) ok = take_row(pb, nb) && ok;
                if (wt) ok = take_row(pt, nt) && ok;
                return ok;
            }))
            return;
        if (wb) vb = nb;
        if (wt) vt = nt;
        if (!(left || right)) return;
        if (wl) sh.face[wave][0][lane] = (unsigned)ql;
        if (wr) sh.face[wave][1][lane] = (unsigned)qr;
        wave_lds_fence();
        if ((lane == 0 && left) || (lane == nout + 1 && right)) {
            const unsigned *f = &sh.face[wave][lane == 0 ? 0 : 1][0];
#pragma unroll
            for (int j = 0; j < R; j++) v[j] = get(f, j);
        }
        wave_lds_fence();
    }

    // All-reduce of NV values: part() with each wave's sums, a barrier,
    // post_total() and collect_total(), a barrier, total().  Wave q collects the
    // sums of workgroups 64 q .. 64 q + 63; every workgroup forms every total
    // in the same order, so all get the same bits.
    template <int NV> __device__ void part(Sh &sh, DD (&acc)[NV]) const
    {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const DD t = wave_reduce(acc[v]);
            if (lane == WAVE - 1) sh.part[v][wave] = t;
        }
    }
    template <int NV> __device__ void post_total(Sh &sh)
    {
        rtag++;
        if (wave != 0) return;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            DD t = lane < RES_WAVES ? sh.part[v][lane] : DD{0.0, 0.0};
            dpp_merge<0x111, 0xf>(t);
            dpp_merge<0x112, 0xf>(t);
            dpp_merge<0x114, 0xf>(t);   // lane 7: the workgroup's sum
            if (nwg == 1) {
                if (lane == RES_WAVES - 1) sh.sum[v][0] = t;
                continue;
            }
            // lane 4 c + k writes word k of copy c
            const word_t sum_s = (word_t)__double_as_longlong(lane_value(t.s, RES_WAVES - 1));
            const word_t sum_c = (word_t)__double_as_longlong(lane_value(t.c, RES_WAVES - 1));
            const word_t half = lane & 2 ? sum_c : sum_s;
            if (lane < 4 * RED_COPIES)
                store_word(red_at(lane / 4, wg, v * 4 + lane % 4), rtag, (unsigned)(lane & 1 ? half >> 32 : half));
        }
    }
    template <int NV, int WAIT = 0> __device__ void collect_total(Sh &sh)
    {
        if (nwg == 1 || wave * WAVE >= nwg) return;
        if (WAIT) __builtin_amdgcn_s_sleep(WAIT);
        const int from = wave * WAVE + lane;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const word_t *p = red_at(wg % RED_COPIES, from, v * 4);
            word_t q[4] = {0, 0, 0, 0};
            if (!poll<NEXT_LOOK>(sh, [&] {
                    if (from >= nwg) return true;
#pragma unroll
                    for (int k = 0; k < 4; k++) q[k] = load_word(p + k * RES_MAX_WG);
                    return (unsigned)(q[0] >> 32) == rtag && (unsigned)(q[1] >> 32) == rtag &&
                           (unsigned)(q[2] >> 32) == rtag && (unsigned)(q[3] >> 32) == rtag;
                }))
                return;
            DD t;
            t.s = __longlong_as_double((long long)((q[0] & 0xffffffffull) | (q[1] << 32)));
            t.c = __longlong_as_double((long long)((q[2] & 0xffffffffull) | (q[3] << 32)));
            t = wave_reduce(t);
            if (lane == WAVE - 1) sh.sum[v][wave] = t;
        }
    }
    __device__ double total(const Sh &sh, int v) const
    {
        DD t = sh.sum[v][0];
        for (int q = 1; q * WAVE < nwg; q++) dd_merge(t, sh.sum[v][q]);
        return t.s + t.c;
    }

    // Waits until try_once() holds in every lane; false (and sh.bad) after
    // EXCHANGE_TICKS, or soon after another wave gave up, so every wait ends.
    template <int GAP = 1, typename F> __device__ bool poll(Sh &sh, F try_once)
    {
        long long t0 = 0;
        for (int spins = 0;; spins++) {
            if (__all(try_once())) return true;
            __builtin_amdgcn_s_sleep(GAP);
            if ((spins & 1023) == 1023) {
                if (__hip_atomic_load(&sh.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) return false;
                const long long now = wall_clock64();
                if (t0 == 0) t0 = now;
                if (now - t0 > EXCHANGE_TICKS) {
                    sh.bad = 1;
                    return false;
                }
            }
        }
    }

    // Every workgroup of the launch is on the chip, or none goes on (one
    // atomic verdict): the exchanges need all of them to make progress.
    __device__ bool start(Sh &sh)
    {
        if (threadIdx.x == 0) {
            sh.bad = 0;
            unsigned verdict = VERDICT_GO;
            if (nwg > 1) {
                const unsigned n = __hip_atomic_fetch_add(&x.ctl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (n == (unsigned)nwg - 1) decide(VERDICT_GO);
                const long long t0 = wall_clock64();
                while ((verdict = __hip_atomic_load(&x.ctl[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ==
                       VERDICT_NONE)
                    if (wall_clock64() - t0 > START_TICKS) decide(VERDICT_ABORT);
            }
            sh.verdict = (int)verdict;
        }
        __syncthreads();
        return sh.verdict == VERDICT_GO;
    }
    // The last workgroup to leave clears the counters for the next launch.
    __device__ void leave()
    {
        if (threadIdx.x == 0 && nwg > 1) {
            const unsigned n = __hip_atomic_fetch_add(&x.ctl[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (n == (unsigned)nwg - 1)
                for (int k = 0; k < 3; k++)
                    __hip_atomic_store(&x.ctl[k], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }

private:
    __device__ void decide(unsigned v)
    {
        unsigned none = VERDICT_NONE;
        __hip_atomic_compare_exchange_strong(&x.ctl[1], &none, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ static void put(unsigned *f, int j, T v)
    {
        if constexpr (sizeof(T) == 4) {
            f[j] = __float_as_uint(v);
        } else {
            const unsigned long long b = (unsigned long long)__double_as_longlong(v);
            f[2 * j] = (unsigned)b;
            f[2 * j + 1] = (unsigned)(b >> 32);
        }
    }
    __device__ static T get(const unsigned *f, int j)
    {
        if constexpr (sizeof(T) == 4) return __uint_as_float(f[j]);
        else return __longlong_as_double((long long)(((unsigned long long)f[2 * j + 1] << 32) | f[2 * j]));
    }
    // word k of workgroup w's sums in a copy: the same word of neighbouring
    // workgroups side by side, so that a wave reads whole lines
    __device__ word_t *red_at(int copy, int w, int k) const
    {
        return x.red + (((size_t)(rtag & 1) * RED_COPIES + copy) * 8 + k) * RES_MAX_WG + w;
    }
    __device__ word_t *col_at(int slot, int w, int side) const
    {
        return x.col + (((size_t)(slot * RES_MAX_WG + w) * 2 + side) * RES_WAVES + wave) * FACE_WORDS + lane;
    }
    __device__ word_t *row_at(int slot, int w, int side) const
    {
        return x.row + ((size_t)(slot * RES_MAX_WG + w) * 2 + side) * 2 * 64 + lane;
    }
    __device__ void post_row(int slot, int side, T v)
    {
        if (!out) return;
        word_t *p = row_at(slot, wg, side);
        if constexpr (sizeof(T) == 4) {
            store_word(p, xtag, __float_as_uint(v));
        } else {
            const unsigned long long b = (unsigned long long)__double_as_longlong(v);
            store_word(p, xtag, (unsigned)b);
            store_word(p + 64, xtag, (unsigned)(b >> 32));
        }
    }
    __device__ bool take_row(const word_t *p, T &v) const
    {
        if constexpr (sizeof(T) == 4) {
            const word_t a = load_word(p);
            v = __uint_as_float((unsigned)a);
            return (unsigned)(a >> 32) == xtag;
        } else {
            const word_t a = load_word(p), b = load_word(p + 64);
            v = __longlong_as_double((long long)((a & 0xffffffffull) | (b << 32)));
            return (unsigned)(a >> 32) == xtag && (unsigned)(b >> 32) == xtag;
        }
    }
};

// The operator's coefficients of a workgroup's rows, in LDS (one column per
// lane): kx[j], ky[j] at row r0 + j, with the face above the last row at
// ky[nrows].  They are read once per product, in registers they would take
// two fifths of what an inner step holds.
template <typename T, int S> struct Coefs {
    static constexpr int R = S * STRIP;
    T kxs[RES_WAVES][R][WAVE], kys[RES_WAVES][R + 1][WAVE];
    __device__ void load(const Place<T, S> &w, const T *Kx, const T *Ky)
    {
        const FieldBuf<T> bx = w.field(Kx), by = w.field(Ky);
#pragma unroll
        for (int k = 0; k < S; k++) {
            T x[STRIP], y[STRIP];
#pragma unroll
            for (int i = 0; i < STRIP; i++) {
                x[i] = w.load(bx, w.o_mem, k * STRIP + i, w.nrows);
                y[i] = w.load(by, w.o_in, k * STRIP + i, w.nrows > 0 ? w.nrows + 1 : 0);
            }
#pragma unroll
            for (int i = 0; i < STRIP; i++) {
                kxs[w.wave][k * STRIP + i][w.lane] = x[i];
                kys[w.wave][k * STRIP + i][w.lane] = y[i];
            }
        }
        kys[w.wave][R][w.lane] = w.load(by, w.o_in, R, w.nrows > 0 ? w.nrows + 1 : 0);
        wave_lds_fence();
    }
    __device__ T kx(const Place<T, S> &w, int j) const { return kxs[w.wave][j][w.lane]; }
    __device__ T ky(const Place<T, S> &w, int j) const { return kys[w.wave][j][w.lane]; }
    __device__ T diag(const Place<T, S> &w, int j) const
    {
        const T k0 = kx(w, j);
        return T(1.0) + (ky(w, j + 1) + ky(w, j)) + (lane_from_above(k0) + k0);
    }
    // (A v) at row j, in the expression order of tea_leaf_cg.cuknl:53-57; v
    // holds the row above the wave's last at v[4 mine], vb is the row below the first
    __device__ T apply(const Place<T, S> &w, const T (&v)[R + 1], T vb, int j) const
    {
        const T kx0 = kx(w, j), kx1 = lane_from_above(kx0), ky0 = ky(w, j), ky1 = ky(w, j + 1);
        const T right = lane_from_above(v[j]), left = lane_from_below(v[j]);
        const T under = j > 0 ? v[j > 0 ? j - 1 : 0] : vb;
        return (T(1.0) + (ky1 + ky0) + (kx1 + kx0)) * v[j] - (ky1 * v[j + 1] + ky0 * under) -
               (kx1 * right + kx0 * left);
    }
};

// The preconditioner of a wave's strips: factors formed once (the expressions
// of init_jac_diag and block_init), one column per lane, in LDS where they fit
// beside the coefficients and in registers where they do not.
template <typename T, int PREC, int S> struct Factors {
    static constexpr int R = S * STRIP;
    // block: cp[0..2], bfp[1..3], diag0 per strip (FP32: 1/diag0 in double in two words)
    static constexpr int PER_STRIP = PREC == PREC_BLOCK ? (sizeof(T) == 4 ? 8 : 7) : (PREC == PREC_DIAG ? STRIP : 0);
    static constexpr int N = PER_STRIP * S;
    static constexpr size_t LDS_BYTES = 160 * 1024;
    static constexpr bool IN_LDS =
        N > 0 && sizeof(T) * RES_WAVES * WAVE * N + sizeof(Coefs<T, S>) + sizeof(Shared<T, S>) +
                         sizeof(T) * RES_WAVES * 2 * R + 256 <= LDS_BYTES;
    struct Store {
        T f[IN_LDS ? RES_WAVES : 1][IN_LDS ? N : 1][IN_LDS ? WAVE : 1];
    };
    T reg[!IN_LDS && N > 0 ? N : 1];
    Store *lds;
    int wave, lane;

    __device__ void put(int k, T v)
    {
        if constexpr (IN_LDS) lds->f[wave][k][lane] = v;
        else if constexpr (N > 0) reg[k] = v;
    }
    __device__ T get(int k) const
    {
        if constexpr (IN_LDS) return lds->f[wave][k][lane];
        else return reg[N > 0 ? k : 0];
    }

    __device__ void init(Store &store, const Place<T, S> &w, const Coefs<T, S> &co)
    {
        lds = &store;
        wave = w.wave;
        lane = w.lane;
        if constexpr (PREC == PREC_DIAG) {
#pragma unroll
            for (int j = 0; j < R; j++) put(j, T(1.0) / co.diag(w, j));
        } else if constexpr (PREC == PREC_BLOCK) {
#pragma unroll
            for (int k = 0; k < S; k++) {
                T d[STRIP], kyk[STRIP + 1], cp[STRIP], bfp[STRIP];
#pragma unroll
                for (int j = 0; j < STRIP; j++) d[j] = co.diag(w, k * STRIP + j);
#pragma unroll
                for (int j = 0; j <= STRIP; j++) kyk[j] = co.ky(w, k * STRIP + j);
                strip_factor(w.strip_len(k), d, kyk, cp, bfp);
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    put(k * PER_STRIP + j, cp[j]);
                    put(k * PER_STRIP + 3 + j, bfp[j + 1]);
                }
                if constexpr (sizeof(T) == 4) {
                    const unsigned long long b = (unsigned long long)__double_as_longlong(1.0 / (double)d[0]);
                    put(k * PER_STRIP + 6, __uint_as_float((unsigned)b));
                    put(k * PER_STRIP + 7, __uint_as_float((unsigned)(b >> 32)));
                } else {
                    put(k * PER_STRIP + 6, d[0]);
                }
            }
        }
    }

    // Mi at row j (jac_diag)
    __device__ T mi(int j) const { return get(j); }

    // z = M^-1 r on strip k
    __device__ void apply(const Place<T, S> &w, const Coefs<T, S> &co, int k, const T (&r)[STRIP],
                          T (&z)[STRIP]) const
    {
        if constexpr (PREC == PREC_NONE) {
#pragma unroll
            for (int j = 0; j < STRIP; j++) z[j] = r[j];
        } else if constexpr (PREC == PREC_DIAG) {
#pragma unroll
            for (int j = 0; j < STRIP; j++) z[j] = r[j] * get(k * STRIP + j);
        } else {
            T cp[STRIP], bfp[STRIP], kyk[STRIP + 1];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                cp[j] = get(k * PER_STRIP + j);
                bfp[j + 1] = get(k * PER_STRIP + 3 + j);
            }
            cp[3] = bfp[0] = T(0.0);
            kyk[0] = kyk[STRIP] = T(0.0);   // (not read)
#pragma unroll
            for (int j = 1; j < STRIP; j++) kyk[j] = co.ky(w, k * STRIP + j);
#pragma unroll
            for (int j = 0; j < STRIP; j++) z[j] = T(0.0);
            if constexpr (sizeof(T) == 4) {
                const unsigned lo = __float_as_uint(get(k * PER_STRIP + 6)), hi = __float_as_uint(get(k * PER_STRIP + 7));
                const double rd = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
                strip_apply_rd(r, z, w.strip_len(k), rd, kyk, cp, bfp);
            } else {
                strip_apply(r, z, w.strip_len(k), get(k * PER_STRIP + 6), kyk, cp, bfp);
            }
        }
    }
};

// The first workgroup copies the run's values to the host's memory when it is
// over: a store across the bus inside the loop would hold up that workgroup's
// next exchange, and with it every other.
__device__ __forceinline__ void report(const Exchange &x, double *history, int n)
{
    __syncthreads();   // thread 0 wrote them
    for (int k = threadIdx.x; k < n; k += RES_BLOCK) history[k] = x.history[k];
}

// A value the compiler takes as new here: offsets derived from it are formed
// where they are used instead of being held across the iterations.
__device__ __forceinline__ unsigned fresh(unsigned o)
{
    asm volatile("" : "+v"(o));
    return o;
}

__device__ __forceinline__ bool replacement_due(const Stop &st, double q_ref, double q)
{
    const double drop = sqrt(fabs(q / q_ref));
    const double predicted = sqrt(fabs(st.rr_ref)) * drop;
    return !(drop >= st.delta && predicted >= st.target);
}

// CG iterations on resident tiles.  Bound by the latency of the two all-reduces
// of an iteration on small meshes and by FP64 issue on the largest that fit.
// u's update runs while the second all-reduce is under way; p, u, r and one
// more column of a strip stay in registers (up to 16 rows in FP64, 32 in FP32:
// 256 registers, two waves per SIMD; one wave per SIMD with 512 registers was
// slower, 11.4 against 9.1 us per iteration of 1000^2 cells, with nothing to
// run while a chain of FP64 operations waits).
// Measured, FP64 without a preconditioner, a deck's whole run with its set-up,
// against the separate kernels: 10^2 cells 1.38 (3.43) ms, 250^2 1.95 (10.15)
// ms, 1000^2 5.18 (25.00) ms; per iteration 6 us at 250^2 (two exchanges'
// latency), 9 at 1000^2 (that and FP64 issue).
template <typename T, int PREC, int S>
__global__ __launch_bounds__(RES_BLOCK, 2) void k_cg_resident(Tiles t, Fields<T> f, Exchange x, int with_p,
                                                              double beta_in, double rro, Stop st, int max_its,
                                                              double *history, Outcome *outcome)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<T, S> sh;
    __shared__ Coefs<T, S> co;
    __shared__ typename Factors<T, PREC, S>::Store fac_store;
    Place<T, S> w(t, x);
    if (!w.start(sh)) {
        if (w.wg == 0 && threadIdx.x == 0) outcome->iterations = -1;
        w.leave();
        return;
    }
    Factors<T, PREC, S> fac;
    co.load(w, f.Kx, f.Ky);
    fac.init(fac_store, w, co);
    const FieldBuf<T> bu = w.field(f.u), br = w.field(f.r), bp = w.field(f.p);
    T u[R], r[R], p[R + 1], pb = T(0.0), v[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        u[j] = w.load(bu, w.o_out, j, w.nrows);
        r[j] = w.load(br, w.o_out, j, w.nrows);
        v[j] = T(0.0);
    }
    const int rows_p = w.nrows > 0 ? w.nrows + 1 : 0;
#pragma unroll
    for (int j = 0; j <= R; j++) p[j] = w.load(bp, w.o_mem, j, rows_p);
    pb = w.load_below(bp, w.o_mem);
    if (with_p) {   // p = z + beta p inside the mesh
        const FieldBuf<T> bz = w.field(PREC == PREC_NONE ? f.r : f.z);
        const T beta = (T)beta_in;
        const int rows_in = w.nrows > 0 ? w.nrows + (w.in_above ? 1 : 0) : 0;
#pragma unroll
        for (int j = 0; j <= R; j++) {
            const T zv = w.load(bz, w.o_in, j, rows_in);
            if (w.col_in && j < rows_in) p[j] = zv + beta * p[j];
        }
        const T zv = w.load_below(bz, w.in_below ? w.o_in : OOB);
        if (w.col_in && w.in_below) pb = zv + beta * pb;
    }
    double q_ref = st.q_ref;
    int have_q = st.have_q, it = 0;
    for (;;) {
        DD acc[1] = {{0.0, 0.0}};
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
#pragma unroll
                for (int i = 0; i < STRIP; i++) v[k * STRIP + i] = co.apply(w, p, pb, k * STRIP + i);
                w.cut(k, v, k * STRIP);
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    const int j = k * STRIP + i;
                    dd_add_prod(acc[0], (double)p[j], (double)v[j]);
                }
            }
        }
        acc[0] = w.owned(acc[0]);
        w.template part<1>(sh, acc);
        __syncthreads();
        w.template post_total<1>(sh);
        w.template collect_total<1, FIRST_LOOK>(sh);
        __syncthreads();
        if (sh.bad) break;
        const double pw = w.total(sh, 0);
        const T alpha = (T)(rro / pw);
        acc[0] = DD{0.0, 0.0};
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
                T rv[STRIP], zv[STRIP];
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    const int j = k * STRIP + i;
                    r[j] = r[j] - alpha * v[j];
                    rv[i] = r[j];
                }
                fac.apply(w, co, k, rv, zv);
                w.cut(k, zv);
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    v[k * STRIP + i] = zv[i];
                    dd_add_prod(acc[0], (double)rv[i], (double)zv[i]);
                }
            }
        }
        acc[0] = w.owned(acc[0]);
        w.post(sh, v);
        w.template part<1>(sh, acc);
        __syncthreads();
        w.template post_total<1>(sh);
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
#pragma unroll
                for (int i = 0; i < STRIP; i++) u[k * STRIP + i] += alpha * p[k * STRIP + i];
            }
        }
        T zb = T(0.0), zt = T(0.0);
        w.take(sh, v, zb, zt);
        w.template collect_total<1>(sh);
        __syncthreads();
        if (sh.bad) break;
        const double rrn = w.total(sh, 0);
        if (w.wg == 0 && threadIdx.x == 0) {
            x.history[2 * it] = pw;
            x.history[2 * it + 1] = rrn;
        }
        it++;
        const double error = sqrt(fabs(rrn));
        bool stop = it >= max_its || error < st.error_below || (it >= st.switch_after && error <= st.switch_error);
        if (st.reliable) {
            if (!have_q) {
                q_ref = rrn;
                have_q = 1;
            } else {
                stop = stop || replacement_due(st, q_ref, rrn);
            }
        }
        if (stop) break;
        const T beta = (T)(rrn / rro);
        rro = rrn;
        if (w.col_in) {
            const T pt = zt + beta * get_top<S>(p, w.mine);
#pragma unroll
            for (int k = 0; k < S; k++) {
                if (k < w.mine) {
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        const int j = k * STRIP + i;
                        p[j] = v[j] + beta * p[j];
                    }
                    w.cut(k, p, k * STRIP);
                }
            }
            if (w.in_above) set_top<S>(p, w.mine, pt);
            if (w.in_below) pb = zb + beta * pb;
        }
    }
    const FieldBuf<T> bz = w.field(f.z);
#pragma unroll
    for (int j = 0; j < R; j++) {
        w.store(bu, w.o_out, j, w.nrows, u[j]);
        w.store(br, w.o_out, j, w.nrows, r[j]);
        w.store(bp, w.o_out, j, w.nrows, p[j]);
        if (PREC != PREC_NONE) w.store(bz, w.o_out, j, w.nrows, v[j]);
    }
    if (w.wg == 0) {
        report(x, history, 2 * it);
        if (threadIdx.x == 0) outcome->iterations = sh.bad ? -2 : it;
    }
    w.leave();
}

// PPCG outer iterations on resident tiles.  The inner steps' fields (sd,
// rtemp, utemp) stay in registers and the coefficients in LDS; p, u, r and
// rstore, which an outer iteration reads once or twice, stay in memory (each
// lane its own cells) but for the smallest tiles, where the registers hold
// them too (more would spill inside the inner steps, and a spill there costs
// more than the reads).  An inner step is one neighbour exchange (no
// all-reduce): bound by its latency on small meshes, by issue on the largest.
// Measured, a deck's whole run with its CG steps and set-up, against the
// separate passes: FP64, 512^2 block Jacobi, 10 inner steps 4.42 (10.50) ms; 1531
// x 997 jac_diag, halo depth 2, to the FP64 true residual 10.64 (20.12) ms (with
// selects per row instead of branches per strip 9% more).  There, four strips
// per wave, two thirds of an inner step are issue and a fifth the exchange, and
// 86 registers spill (152 with block Jacobi: 1400^2 8.4 (15.9) ms).  FP32 block
// Jacobi: 1000^2, 3 strips, 4.5 (8.3) ms; 1980^2, 8 strips, 19.9 (24.2) ms.
template <typename T, int PREC, int S>
__global__ __launch_bounds__(RES_BLOCK, 2) void k_ppcg_resident(Tiles t, Fields<T> f, Exchange x, int from_inner,
                                                                int with_p, double beta_in, double rro,
                                                                double theta_in, const double *__restrict__ coef,
                                                                int coef_stride, int steps, Stop st, int max_its,
                                                                double *history, Outcome *outcome)
{
    constexpr int R = S * STRIP;
    constexpr bool KEEP = R * sizeof(T) <= 32;   // p, u, r and rstore in registers too
    constexpr int RK = KEEP ? R : 1;
    __shared__ Shared<T, S> sh;
    __shared__ Coefs<T, S> co;
    __shared__ typename Factors<T, PREC, S>::Store fac_store;
    __shared__ T halo_p[KEEP ? 1 : RES_WAVES][2][R];   // p of the halo lanes between outer iterations
    Place<T, S> w(t, x);
    if (!w.start(sh)) {
        if (w.wg == 0 && threadIdx.x == 0) outcome->iterations = -1;
        w.leave();
        return;
    }
    Factors<T, PREC, S> fac;
    co.load(w, f.Kx, f.Ky);
    fac.init(fac_store, w, co);
    const FieldBuf<T> bu = w.field(f.u), br = w.field(f.r), bp = w.field(f.p), brs = w.field(f.rstore);
    const T theta_r = T(1.0) / (T)theta_in;
    const bool halo_lane = w.lane == 0 || w.lane == w.nout + 1;
    T sd[R + 1], rt[R], ut[R + 1], utb = T(0.0), sdb = T(0.0), pb, pt;
    // z of the first begin, and p's halo
#pragma unroll
    for (int j = 0; j <= R; j++) ut[j] = T(0.0);
    if (with_p || !from_inner) {
        const FieldBuf<T> bz = w.field(f.z_in);
        const int rows_in = w.nrows > 0 ? w.nrows + (w.in_above ? 1 : 0) : 0;
#pragma unroll
        for (int j = 0; j <= R; j++) ut[j] = w.load(bz, w.o_in, j, rows_in);
        utb = w.load_below(bz, w.in_below ? w.o_in : OOB);
    }
    const int rows_p = w.nrows > 0 ? w.nrows + 1 : 0;
    pb = w.load_below(bp, w.o_mem);
    pt = bp.load(w.nrows > 0 ? w.o_mem : OOB, (unsigned)w.nrows * w.row_b);
    T pk[RK], uk[RK], rk[RK], rsk[RK];
    const int rows_s = w.nrows % STRIP ? rows_p : w.nrows;   // with the row above a strip cut short: its p never changes
    if (KEEP) {
#pragma unroll
        for (int j = 0; j < RK; j++) {
            pk[j] = w.load(bp, w.o_mem, j, rows_s);
            uk[j] = w.load(bu, w.o_out, j, w.nrows);
            rk[j] = w.load(br, w.o_out, j, w.nrows);
            rsk[j] = w.load(brs, w.o_out, j, w.nrows);
        }
    } else {
        T hp[R];
#pragma unroll
        for (int j = 0; j < R; j++) hp[j] = w.load(bp, halo_lane ? w.o_mem : OOB, j, w.nrows);
        if (halo_lane) {
#pragma unroll
            for (int j = 0; j < R; j++) halo_p[w.wave][w.lane == 0 ? 0 : 1][j] = hp[j];
        }
        wave_lds_fence();
    }
    double q_ref = st.q_ref, beta_now = beta_in, rz = rro, pw = 0.0;
    int have_q = st.have_q, it = 0, at_ur = 0;
    bool inner_first = from_inner != 0;
    double rrn_end = 0.0;
    for (;;) {
        DD acc[2] = {{0.0, 0.0}, {0.0, 0.0}};
        T alpha = T(0.0);
        if (!inner_first) {
            // ---- begin: p = z + beta p (in sd), w = A p (in rt), rstore = r
            const T beta = (T)beta_now;
            const unsigned o = fresh(w.o_out), om = fresh(w.o_mem);
            sd[R] = T(0.0);
#pragma unroll
            for (int j = 0; j < R; j++) {
                sd[j] = KEEP ? pk[KEEP ? j : 0] : w.load(bp, om, j, rows_s);
                rt[j] = KEEP ? rk[KEEP ? j : 0] : w.load(br, o, j, w.nrows);   // r
            }
#pragma unroll
            for (int j = 0; j < R; j++) {
                if (!KEEP && halo_lane && j < w.nrows) sd[j] = halo_p[w.wave][w.lane == 0 ? 0 : 1][j];
                dd_add_prod(acc[1], (double)rt[j], w.out && j < w.nrows ? (double)ut[j] : 0.0);
                if (with_p && w.col_in && j < w.nrows) sd[j] = ut[j] + beta * sd[j];
            }
            if (with_p && w.col_in) {
                if (w.in_above) pt = get_top<S>(ut, w.mine) + beta * pt;
                if (w.in_below) pb = utb + beta * pb;
            }
            if (w.nrows % STRIP == 0) set_top<S>(sd, w.mine, pt);
#pragma unroll
            for (int j = 0; j < R; j++) ut[j] = rt[j];   // r
    #pragma unroll
            for (int k = 0; k < S; k++) {
                if (k < w.mine) {
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        const int j = k * STRIP + i;
                        const T a = co.apply(w, sd, pb, j);
                        rt[j] = w.out && j < w.nrows ? a : T(0.0);
                        dd_add_prod(acc[0], (double)sd[j], (double)rt[j]);
                    }
                }
            }
            w.template part<2>(sh, acc);
            __syncthreads();
            w.template post_total<2>(sh);
            // while the sums travel: rstore = r
#pragma unroll
            for (int j = 0; j < R; j++) {
                if (KEEP) {
                    pk[KEEP ? j : 0] = sd[j];
                    rsk[KEEP ? j : 0] = ut[j];
                } else {
                    w.store(brs, o, j, w.nrows, ut[j]);
                }
            }
            if (!KEEP && halo_lane) {
#pragma unroll
                for (int j = 0; j < R; j++) halo_p[w.wave][w.lane == 0 ? 0 : 1][j] = sd[j];
            }
            w.template collect_total<2>(sh);
            __syncthreads();
            if (sh.bad) break;
            // p goes to memory only now: the neighbours read its outer cells there
            // when their run starts, and their sums, which have come, follow those reads
            if (!KEEP) {
#pragma unroll
                for (int j = 0; j < R; j++) w.store(bp, o, j, w.nrows, sd[j]);
            }
            pw = w.total(sh, 0);
            rz = w.total(sh, 1);
            alpha = (T)(rz / pw);
        } else {
#pragma unroll
            for (int j = 0; j < R; j++) {
                ut[j] = KEEP ? rk[KEEP ? j : 0] : w.load(br, w.o_out, j, w.nrows);
                rt[j] = T(0.0);
            }
        }
        // ---- ur: r -= alpha w, z = M^-1 r, r.z; sd = z / theta, rtemp = r, utemp = sd
        acc[0] = DD{0.0, 0.0};
        const unsigned o_ur = fresh(w.o_out);
#pragma unroll
        for (int j = 0; j < R; j++) {
            if (j >= w.mine * STRIP) {
                sd[j] = rt[j] = ut[j] = T(0.0);
            }
        }
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
                T rv[STRIP], zv[STRIP];
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    const int j = k * STRIP + i;
                    rv[i] = ut[j];
                    if (!inner_first) {
                        rv[i] = rv[i] - alpha * rt[j];
                        if (KEEP) {
                            rk[KEEP ? j : 0] = rv[i];
                            uk[KEEP ? j : 0] += alpha * pk[KEEP ? j : 0];
                        } else {
                            w.store(br, o_ur, j, w.nrows, rv[i]);
                        }
                    }
                }
                fac.apply(w, co, k, rv, zv);
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    const int j = k * STRIP + i;
                    const T z = w.out && j < w.nrows ? zv[i] : T(0.0);
                    dd_add_prod(acc[0], (double)rv[i], (double)z);
                    sd[j] = z * theta_r;
                    rt[j] = rv[i];
                    ut[j] = sd[j];
                }
            }
        }
        // ---- inner steps; the exchange of the latest sd comes first
        for (int s = 0;; s++) {
            T sdt = T(0.0);
            sdb = T(0.0);
            w.post(sh, sd);
            __syncthreads();
            // u += alpha p, a strip per step while the exchange is under way (the rest in the last)
            if (!KEEP && !inner_first) {
                for (int k = s; k < w.mine && (k == s || s == steps); k++) {
                    const unsigned o = fresh(w.o_out);
                    T un[STRIP], pn[STRIP];
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        un[i] = w.load(bu, o, k * STRIP + i, w.nrows);
                        pn[i] = w.load(bp, o, k * STRIP + i, w.nrows);
                    }
#pragma unroll
                    for (int i = 0; i < STRIP; i++)
                        w.store(bu, o, k * STRIP + i, w.nrows, un[i] + alpha * pn[i]);
                }
            }
            w.take(sh, sd, sdb, sdt);
            set_top<S>(sd, w.mine, sdt);
            // utemp of the halo: the same sums as the neighbour's
            if (s == 0) {
                utb = sdb;
                set_top<S>(ut, w.mine, sdt);
            } else {
                utb += sdb;
                set_top<S>(ut, w.mine, get_top<S>(ut, w.mine) + sdt);
            }
            if (halo_lane && s == 0) {
                asm volatile("" ::: "memory");   // (branches, as below; rows beyond the wave's are of no use)
#pragma unroll
                for (int j = 0; j < R; j++) ut[j] = sd[j];
            } else if (halo_lane) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < R; j++) ut[j] += sd[j];
            }
            if (s == steps) break;
            const T a = (T)coef[s], b = (T)coef[coef_stride + s];
    #pragma unroll
            for (int k = 0; k < S; k++) {
                if (k < w.mine) {
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        const int j = k * STRIP + i;
                        rt[j] = rt[j] - co.apply(w, sd, sdb, j);   // (of no use outside the tile, but harmless)
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < S; k++) {
                if (k < w.mine) {
                    T rv[STRIP], nv[STRIP];
#pragma unroll
                    for (int i = 0; i < STRIP; i++) rv[i] = rt[k * STRIP + i];
                    if (PREC == PREC_BLOCK) {
                        T zv[STRIP];
                        fac.apply(w, co, k, rv, zv);
#pragma unroll
                        for (int i = 0; i < STRIP; i++) nv[i] = a * sd[k * STRIP + i] + b * zv[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < STRIP; i++) {
                            const int j = k * STRIP + i;
                            if (PREC == PREC_DIAG) nv[i] = a * sd[j] + b * rv[i] * fac.mi(j);
                            else nv[i] = a * sd[j] + b * rv[i];
                        }
                    }
                    w.cut(k, nv);
                    if (w.out) {
                        asm volatile("" ::: "memory");   // one branch per strip, not selects on every row
#pragma unroll
                        for (int i = 0; i < STRIP; i++) {
                            const int j = k * STRIP + i;
                            sd[j] = nv[i];
                            ut[j] += nv[i];
                        }
                    }
                }
            }
        }
        // ---- end: z = utemp, (r - rstore).z (sd and rtemp, which a run that ends
        // here still writes out, are kept while rstore and r come in)
        acc[1] = DD{0.0, 0.0};
        const unsigned o_end = fresh(w.o_out);
#pragma unroll
        for (int k = 0; k < S; k++) {
            T rv[STRIP], rs[STRIP];
#pragma unroll
            for (int i = 0; i < STRIP; i++) {
                rv[i] = KEEP ? rk[KEEP ? k * STRIP + i : 0] : w.load(br, o_end, k * STRIP + i, w.nrows);
                rs[i] = KEEP ? rsk[KEEP ? k * STRIP + i : 0] : w.load(brs, o_end, k * STRIP + i, w.nrows);
            }
#pragma unroll
            for (int i = 0; i < STRIP; i++) {
                const int j = k * STRIP + i;
                const T d = rv[i] - rs[i];
                dd_add_prod(acc[1], (double)d, w.out && j < w.nrows ? (double)ut[j] : 0.0);
            }
        }
        w.template part<2>(sh, acc);
        __syncthreads();
        w.template post_total<2>(sh);
        w.template collect_total<2>(sh);
        __syncthreads();
        if (sh.bad) break;
        const double rrn_ur = w.total(sh, 0), end = w.total(sh, 1);
        bool stop = false;
        if (!inner_first) {
            if (w.wg == 0 && threadIdx.x == 0) {
                x.history[4 * it] = pw;
                x.history[4 * it + 1] = rz;
                x.history[4 * it + 2] = rrn_ur;
                x.history[4 * it + 3] = end;
            }
            it++;
            if (st.reliable) {
                if (!have_q) {
                    q_ref = rrn_ur;
                    have_q = 1;
                } else if (replacement_due(st, q_ref, rrn_ur)) {
                    at_ur = 1;
                    break;
                }
            }
            stop = sqrt(fabs(end)) < st.error_below;
        }
        rrn_end = end;
        inner_first = false;
        if (stop || it >= max_its) break;
        if (PREC == PREC_NONE && st.reliable) {   // the next iteration may end at its ur, which leaves z alone
            const FieldBuf<T> bz = w.field(f.z);
#pragma unroll
            for (int j = 0; j < R; j++) w.store(bz, o_end, j, w.nrows, ut[j]);
        }
        beta_now = rrn_end / rz;
        with_p = 1;
    }
    if (KEEP) {
#pragma unroll
        for (int j = 0; j < RK; j++) {
            w.store(bp, w.o_out, j, w.nrows, pk[j]);
            w.store(bu, w.o_out, j, w.nrows, uk[j]);
            w.store(br, w.o_out, j, w.nrows, rk[j]);
            w.store(brs, w.o_out, j, w.nrows, rsk[j]);
        }
    }
    const FieldBuf<T> bz = w.field(f.z), bsd = w.field(f.sd), brt = w.field(f.rtemp), but = w.field(f.utemp);
    if (at_ur) {   // z = M^-1 r and sd = z / theta again: the inner steps went on for nothing
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
                T rv[STRIP], zv[STRIP];
#pragma unroll
                for (int i = 0; i < STRIP; i++)
                    rv[i] = KEEP ? rk[KEEP ? k * STRIP + i : 0] : w.load(br, w.o_out, k * STRIP + i, w.nrows);
                fac.apply(w, co, k, rv, zv);
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    if (PREC != PREC_NONE) w.store(bz, w.o_out, k * STRIP + i, w.nrows, zv[i]);
                    w.store(bsd, w.o_out, k * STRIP + i, w.nrows, zv[i] * theta_r);
                }
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < R; j++) {
            w.store(bsd, w.o_out, j, w.nrows, sd[j]);
            w.store(brt, w.o_out, j, w.nrows, rt[j]);
            w.store(but, w.o_out, j, w.nrows, ut[j]);
        }
    }
    if (w.wg == 0) {
        report(x, history, 4 * it);
        if (threadIdx.x == 0) {
            outcome->iterations = sh.bad ? -2 : it;
            outcome->at_ur = at_ur;
            outcome->rrn_end = rrn_end;
        }
    }
    w.leave();
}

// Chebyshev iterations on resident tiles: w = A u, r = u0 - w, p = alpha p +
// beta M^-1 r, u += p; one neighbour exchange each, and an all-reduce only in
// the iterations whose norm the caller tests.  w and r are written out where
// the run may end (the reference leaves the last iteration's in their fields).
// Measured, FP64, 1533 x 1021 cells, a deck's whole run with its CG steps and
// set-up, against the separate passes: 4.11 (14.19) ms.
template <typename T, int PREC, int S>
__global__ __launch_bounds__(RES_BLOCK, 2) void k_cheby_resident(Tiles t, Fields<T> f, Exchange x,
                                                                 const double *__restrict__ coef, int coef_stride,
                                                                 int n, int check_from, double error, double target,
                                                                 int max_its, double *history, Outcome *outcome)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<T, S> sh;
    __shared__ Coefs<T, S> co;
    __shared__ typename Factors<T, PREC, S>::Store fac_store;
    Place<T, S> w(t, x);
    if (!w.start(sh)) {
        if (w.wg == 0 && threadIdx.x == 0) outcome->iterations = -1;
        w.leave();
        return;
    }
    Factors<T, PREC, S> fac;
    co.load(w, f.Kx, f.Ky);
    fac.init(fac_store, w, co);
    const FieldBuf<T> bu = w.field(f.u), br = w.field(f.r), bp = w.field(f.p), b0 = w.field(f.u0), bw = w.field(f.w);
    T u[R + 1], p[R], u0[R], v[R], ub;
    const int rows_u = w.nrows > 0 ? w.nrows + 1 : 0;
#pragma unroll
    for (int j = 0; j <= R; j++) u[j] = w.load(bu, w.o_mem, j, rows_u);
    ub = w.load_below(bu, w.o_mem);
#pragma unroll
    for (int j = 0; j < R; j++) {
        p[j] = w.load(bp, w.o_out, j, w.nrows);
        u0[j] = w.load(b0, w.o_out, j, w.nrows);
        v[j] = T(0.0);
    }
    int it = 0;
    for (;; n++) {
        const T alpha = (T)coef[it], beta = (T)coef[coef_stride + it];
        const bool check = n >= check_from && n % 10 == 0;
        const bool last = it + 1 >= max_its || (!check && fabs(sqrt(fabs(error))) < target);
        DD acc[1] = {{0.0, 0.0}};
        const unsigned o = fresh(w.o_out);
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
#pragma unroll
                for (int i = 0; i < STRIP; i++) {
                    const int j = k * STRIP + i;
                    const T a = co.apply(w, u, ub, j);
                    v[j] = u0[j] - a;
                    if (check || last) {
                        w.store(bw, o, j, w.nrows, a);
                        w.store(br, o, j, w.nrows, v[j]);
                    }
                }
                w.cut(k, v, k * STRIP);
            }
        }
        if (check) {
#pragma unroll
            for (int j = 0; j < R; j++) dd_add_prod(acc[0], (double)v[j], (double)v[j]);
            acc[0] = w.owned(acc[0]);
        }
#pragma unroll
        for (int k = 0; k < S; k++) {
            if (k < w.mine) {
                T rv[STRIP], pv[STRIP];
#pragma unroll
                for (int i = 0; i < STRIP; i++) rv[i] = v[k * STRIP + i];
                if (PREC == PREC_BLOCK) {
                    T zv[STRIP];
                    fac.apply(w, co, k, rv, zv);
#pragma unroll
                    for (int i = 0; i < STRIP; i++) pv[i] = alpha * p[k * STRIP + i] + beta * zv[i];
                } else {
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        const int j = k * STRIP + i;
                        if (PREC == PREC_DIAG) pv[i] = alpha * p[j] + beta * fac.mi(j) * rv[i];
                        else pv[i] = alpha * p[j] + beta * rv[i];
                    }
                }
                w.cut(k, pv);
                if (w.out) {
                    asm volatile("" ::: "memory");   // one branch per strip, not selects on every row
#pragma unroll
                    for (int i = 0; i < STRIP; i++) {
                        const int j = k * STRIP + i;
                        p[j] = pv[i];
                        u[j] += pv[i];
                    }
                }
            }
        }
        T ut = get_top<S>(u, w.mine);
        w.post(sh, u);
        if (check) w.template part<1>(sh, acc);
        __syncthreads();
        if (check) w.template post_total<1>(sh);
        w.take(sh, u, ub, ut);
        set_top<S>(u, w.mine, ut);
        if (check) {
            w.template collect_total<1>(sh);
            __syncthreads();
            error = w.total(sh, 0);
        }
        if (w.wg == 0 && threadIdx.x == 0) x.history[it] = check ? error : 0.0;
        it++;
        error = sqrt(fabs(error));
        // (sh.bad only where a barrier has made it the same for all waves)
        if ((check && sh.bad) || it >= max_its || fabs(error) < target) break;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; j++) {
        w.store(bu, w.o_out, j, w.nrows, u[j]);
        w.store(bp, w.o_out, j, w.nrows, p[j]);
    }
    if (w.wg == 0) {
        report(x, history, it);
        if (threadIdx.x == 0) outcome->iterations = sh.bad ? -2 : it;
    }
    w.leave();
}

// Picks the kernel of a preconditioner and number of strips.
#define RESIDENT_PICK(KERNEL, ...)                                                                       \
    do {                                                                                                 \
        const dim3 grid((unsigned)(t.nbx * t.nby)), block(RES_BLOCK);                                    \
        auto go = [&](auto s_c) {                                                                        \
            constexpr int S = decltype(s_c)::value;                                                      \
            if (prec == PREC_BLOCK)                                                                      \
                hipLaunchKernelGGL((KERNEL<T, PREC_BLOCK, S>), grid, block, 0, stream, __VA_ARGS__);     \
            else if (prec == PREC_DIAG)                                                                  \
                hipLaunchKernelGGL((KERNEL<T, PREC_DIAG, S>), grid, block, 0, stream, __VA_ARGS__);      \
            else                                                                                         \
                hipLaunchKernelGGL((KERNEL<T, PREC_NONE, S>), grid, block, 0, stream, __VA_ARGS__);      \
        };                                                                                               \
        switch (t.s) {                                                                                   \
        case 1: go(std::integral_constant<int, 1>{}); break;                                             \
        case 2: go(std::integral_constant<int, 2>{}); break;                                             \
        case 3: go(std::integral_constant<int, 3>{}); break;                                             \
        case 4: go(std::integral_constant<int, 4>{}); break;                                             \
        case 6:                                                                                          \
            if constexpr (sizeof(T) == 4) go(std::integral_constant<int, 6>{});                          \
            break;                                                                                       \
        case 8:                                                                                          \
            if constexpr (sizeof(T) == 4) go(std::integral_constant<int, 8>{});                          \
            break;                                                                                       \
        }                                                                                                \
    } while (0)

}  // namespace

bool plan_tiles(Tiles &t, int nx, int ny, int h, long pitch, int bits, int max_wg)
{
    if (max_wg > RES_MAX_WG) max_wg = RES_MAX_WG;
    if ((double)pitch * (ny + 2.0 * h) * (bits / 8) >= 4294967296.0 - 65536.0) return false;   // 32-bit offsets
    t.e = Ext{h, h + nx - 1, h, h + ny - 1};
    t.pitch = pitch;
    t.nbx = (nx + RES_OUT_X - 1) / RES_OUT_X;
    t.ow = (nx + t.nbx - 1) / t.nbx;
    t.nbx = (nx + t.ow - 1) / t.ow;
    if (t.nbx > max_wg) return false;
    // as many tiles as there are compute units, but none of fewer than 4 strips (one wave per SIMD)
    const int nstrips = (ny + STRIP - 1) / STRIP;
    t.nby = std::min(max_wg / t.nbx, (nstrips + 3) / 4);
    t.ts = (nstrips + t.nby - 1) / t.nby;
    t.nby = (nstrips + t.ts - 1) / t.ts;
    const int need = (t.ts + RES_WAVES - 1) / RES_WAVES;
    for (int s : {1, 2, 3, 4, 6, 8}) {
        if (s > (bits == 32 ? 8 : 4)) break;
        if (s < need) continue;
        t.s = s;
        return true;
    }
    return false;
}

template <typename T>
hipError_t launch_cg(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, int with_p, double beta,
                     double rro, const Stop &st, int max_its, double *history, Outcome *out, hipStream_t stream)
{
    RESIDENT_PICK(k_cg_resident, t, f, x, with_p, beta, rro, st, max_its, history, out);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_ppcg(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, int from_inner, int with_p,
                       double beta, double rro, double theta, const double *coef, int coef_stride, int steps,
                       const Stop &st, int max_its, double *history, Outcome *out, hipStream_t stream)
{
    RESIDENT_PICK(k_ppcg_resident, t, f, x, from_inner, with_p, beta, rro, theta, coef, coef_stride, steps, st, max_its,
                  history, out);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_cheby(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, const double *coef,
                        int coef_stride, int n, int check_from, double error, double target, int max_its,
                        double *history, Outcome *out, hipStream_t stream)
{
    RESIDENT_PICK(k_cheby_resident, t, f, x, coef, coef_stride, n, check_from, error, target, max_its, history, out);
    return hipGetLastError();
}

#define RESIDENT_INSTANCE(T)                                                                                          \
    template hipError_t launch_cg<T>(const Tiles &, int, const Fields<T> &, const Exchange &, int, double, double,    \
                                     const Stop &, int, double *, Outcome *, hipStream_t);                            \
    template hipError_t launch_ppcg<T>(const Tiles &, int, const Fields<T> &, const Exchange &, int, int, double,     \
                                       double, double, const double *, int, int, const Stop &, int, double *,         \
                                       Outcome *, hipStream_t);                                                       \
    template hipError_t launch_cheby<T>(const Tiles &, int, const Fields<T> &, const Exchange &, const double *, int, \
                                        int, int, double, double, int, double *, Outcome *, hipStream_t);
RESIDENT_INSTANCE(double)
RESIDENT_INSTANCE(float)

}  // namespace res
}  // namespace tea
