// Runs k_ppcg_resident's source on the CPU (see hip/hip_runtime.h).
// resident_kernels.inc: csrc/resident.hip up to its launches, and plan_tiles.
#include <ucontext.h>
#include <sys/mman.h>

#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include <hip/hip_runtime.h>

GridDim gridDim;

namespace wavefront {
constexpr int LANES = 512, WAVES_WG = LANES / 64;
constexpr size_t STACK = 128 * 1024;

struct Fibre {
    ucontext_t context;
    Index index;
    enum { READY, MEETING, BARRIER, DONE } state = READY;
    bool paused = false;
};
struct Wave {
    int arrived = 0, turn = 0;
    int values[2][64];
};
struct Workgroup {
    std::vector<Fibre> lanes{LANES};
    Wave waves[WAVES_WG];
    int at_barrier = 0, running = 0;
    ucontext_t scheduler;
    char *stacks = nullptr;
};
thread_local Workgroup *wg;
thread_local Index block;
thread_local std::function<void()> *body;

void fail(const char *what)
{
    fprintf(stderr, "wavefront: %s\n", what);
    abort();
}
const Index &thread_index() { return wg->lanes[wg->running].index; }
static void back() { Fibre &f = wg->lanes[wg->running]; swapcontext(&f.context, &wg->scheduler); }

const int *meet(int value)
{
    const int me = wg->running, l = me & 63;
    Wave &w = wg->waves[me / 64];
    int *values = w.values[w.turn];
    values[l] = value;
    if (++w.arrived == 64) {
        w.arrived = 0;
        w.turn ^= 1;   // a lane that goes on writes the other array
        for (int k = me & ~63; k < (me & ~63) + 64; k++) wg->lanes[k].state = Fibre::READY;
    } else {
        wg->lanes[me].state = Fibre::MEETING;
        back();
    }
    return values;
}
void workgroup_barrier()
{
    if (++wg->at_barrier == LANES) {
        wg->at_barrier = 0;
        for (Fibre &f : wg->lanes) f.state = Fibre::READY;
    } else {
        wg->lanes[wg->running].state = Fibre::BARRIER;
        back();
    }
}
void pause()
{
    wg->lanes[wg->running].paused = true;
    back();
}

// One workgroup at a time: whose turn it is.
struct Turns {
    std::mutex m;
    std::condition_variable cv;
    std::vector<int> order;
    std::vector<bool> over;
    size_t at = 0;
    long idle = 0;
    void next()
    {
        for (size_t k = 0; k < order.size(); k++) {
            at = (at + 1) % order.size();
            if (!over[order[at]]) break;
        }
    }
};

static void lane_main()
{
    (*body)();
    wg->lanes[wg->running].state = Fibre::DONE;
    back();
}

static void run_workgroup(int id, std::function<void()> kernel, Turns &turns)
{
    Workgroup mine;
    wg = &mine;
    block.x = (unsigned)id;
    body = &kernel;
    mine.stacks = (char *)mmap(nullptr, LANES * STACK, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (mine.stacks == MAP_FAILED) fail("no memory for the lanes");
    for (int k = 0; k < LANES; k++) {
        Fibre &f = mine.lanes[k];
        f.index.x = (unsigned)k;
        getcontext(&f.context);
        f.context.uc_stack.ss_sp = mine.stacks + k * STACK;
        f.context.uc_stack.ss_size = STACK;
        f.context.uc_link = nullptr;
        makecontext(&f.context, lane_main, 0);
    }
    for (;;) {
        std::unique_lock<std::mutex> lock(turns.m);
        turns.cv.wait(lock, [&] { return turns.order[turns.at] == id; });
        bool left = true, any = false;
        while (left) {   // until every lane waits for another workgroup or is done
            bool moved = false;
            left = false;
            for (int k = 0; k < LANES; k++) {
                Fibre &f = mine.lanes[k];
                if (f.state != Fibre::READY) continue;
                f.paused = false;
                mine.running = k;
                swapcontext(&mine.scheduler, &f.context);
                if (!f.paused) moved = any = true;
            }
            left = moved;
        }
        bool over = true;
        for (Fibre &f : mine.lanes) over = over && f.state == Fibre::DONE;
        turns.idle = any ? 0 : turns.idle + 1;
        if (turns.idle > 100000) fail("no workgroup gets on");
        if (over) turns.over[id] = true;
        turns.next();
        turns.cv.notify_all();
        if (over) break;
    }
    munmap(mine.stacks, LANES * STACK);
}

// order[k]: the k-th workgroup to run
void launch(int workgroups, const int *order, std::function<void()> kernel)
{
    Turns turns;
    turns.order.assign(order, order + workgroups);
    turns.over.assign(workgroups, false);
    gridDim.x = (unsigned)workgroups;
    std::vector<std::thread> threads;
    for (int k = 0; k < workgroups; k++) threads.emplace_back(run_workgroup, k, kernel, std::ref(turns));
    for (std::thread &t : threads) t.join();
}
}  // namespace wavefront

#include "resident_kernels.inc"

using namespace tea;

// fields: u, p, r, z, Kx, Ky, rstore, sd, rtemp, utemp.  Returns the
// iterations, or -1000 where the plan has another number of strips per wave.
extern "C" int ppcg_resident(int prec, int nx, int ny, int h, int max_wg, const int *order, double **fields,
                             int with_p, double beta, double rro, double theta, const double *coef, int steps,
                             int max_its, double *history, int *at_ur, double *rrn_end, int *tiles_xy)
{
    constexpr int S = 2;
    res::Tiles t;
    if (!res::plan_tiles(t, nx, ny, h, nx + 2 * h, 64, max_wg) || t.s != S) return -1000;
    tiles_xy[0] = t.nbx;
    tiles_xy[1] = t.nby;
    std::vector<res::word_t> words(res::EXCHANGE_WORDS, 0);
    std::vector<double> x_history(4 * res::RES_HISTORY);
    res::Exchange x{};
    x.ctl = (unsigned *)words.data();
    x.red = words.data() + 16;
    x.col = x.red + res::RED_WORDS;
    x.row = x.col + res::COL_WORDS;
    x.history = x_history.data();
    res::Fields<double> f{};
    f.u = fields[0];
    f.p = fields[1];
    f.r = fields[2];
    f.z = fields[3];
    f.z_in = fields[3];
    f.Kx = fields[4];
    f.Ky = fields[5];
    f.rstore = fields[6];
    f.sd = fields[7];
    f.rtemp = fields[8];
    f.utemp = fields[9];
    res::Stop st{};
    st.error_below = -1.0;
    st.switch_after = 1000000000;
    st.switch_error = -1.0;
    res::Outcome out{};
    auto run = [&](auto prec_c) {
        wavefront::launch(t.nbx * t.nby, order, [&] {
            res::k_ppcg_resident<double, decltype(prec_c)::value, S>(t, f, x, 0, with_p, beta, rro, theta, coef,
                                                                    steps, steps, st, max_its, history, &out);
        });
    };
    if (prec == PREC_BLOCK) run(std::integral_constant<int, PREC_BLOCK>{});
    else if (prec == PREC_DIAG) run(std::integral_constant<int, PREC_DIAG>{});
    else run(std::integral_constant<int, PREC_NONE>{});
    *at_ur = out.at_ur;
    *rrn_end = out.rrn_end;
    return out.iterations;
}
