// The host side of the one-launch tolerance solve (resident.hip): which
// cloths of a batch it takes, their parts, and the launch.
#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <stdexcept>

#include "batch.h"

namespace bw
{

namespace
{
void check(hipError_t e, const char *what)
{
    if (e != hipSuccess)
        throw std::runtime_error(std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
}

int env_int(const char *name, int otherwise)
{
    const char *e = std::getenv(name);
    return e ? std::atoi(e) : otherwise;
}

// Limit of a cloth that is solved in one launch, such that any cloths within
// it and RS_SETS_CAP fit a launch's LDS together (resident_lds): rows of
// other parts that a part reads.
int halo_cap(bool fp32) { return fp32 ? RS_HALO32 : RS_HALO64; }
// Parts of a cloth: one per CU (resident_capacity is asked before a launch)
constexpr int PARTS_CAP = 256;
// Iterations that one launch may take (a launch is not interrupted)
constexpr int ITER_CAP = 1000000;

} // namespace

struct ResidentSeats::Device
{
    std::mutex mu;
    std::condition_variable cv;
    int cus = 0, used = 0;
    long long next = 0, serving = 0; // the queue
};

void ResidentSeats::take(int n)
{
    static Device devices[64];
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    Device &d = devices[dev & 63];
    std::unique_lock<std::mutex> lk(d.mu);
    if (d.cus == 0)
        check(hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev),
              "hipDeviceGetAttribute");
    n = std::min(n, d.cus);
    const long long place = d.next++;
    d.cv.wait(lk, [&] { return d.serving == place && d.used + n <= d.cus; });
    d.serving++;
    d.used += n;
    of_ = &d;
    n_ = n;
    d.cv.notify_all(); // the next in the queue may fit too
}

void ResidentSeats::give()
{
    if (!of_)
        return;
    std::lock_guard<std::mutex> lk(of_->mu);
    of_->used -= n_;
    of_->cv.notify_all();
    of_ = nullptr;
}

int resident_extra(bool fp32, int sets_max, int halo_max, int wanted)
{
    const size_t used = resident_lds(fp32, sets_max, halo_max, 0);
    return std::min(wanted, (int)((RS_LDS_MAX - used) / resident_slot_bytes(fp32)));
}

void resident_limits(ResidentLaunch &a, ResidentCtl &ctl, bool w64_leaves)
{
    ctl.wait_ticks = 100000ULL * (unsigned)std::max(0, env_int("BW_RESIDENT_WAIT_MS", 2000));
    a.give_up = env_int("BW_RESIDENT_GIVE_UP", w64_leaves ? -1 : 0);
}

// Parts of each cloth that fits: its slices in order, as many to a
// workgroup as it holds.  BW_RESIDENT=0 turns one-launch solves off;
// BW_GROUP_MIN leaves the cloths above it to the launches, whose order of sums
// it fixes.
Batch::ResidentLists Batch::plan_resident(const std::vector<int> &col,
                                          const std::vector<int> &slice_off,
                                          const std::vector<int> &slice_w,
                                          const std::vector<InstParams> &params)
{
    const bool fp32 = kind_ == SolverKind::CG32;
    const int hold = resident_slices(fp32);
    ResidentPlan &rp = resident_;
    rp = ResidentPlan();
    rp.first.assign(size(), 0);
    rp.count.assign(size(), 0);
    ResidentLists lists;
    std::vector<ResidentPart> &part = lists.part;
    std::vector<int> &halo_row = lists.halo_row, rows;
    std::vector<uint16_t> &pos = lists.pos;
    // (words are addressed by 32-bit byte offsets)
    if (!opt_.one_launch || kind_ == SolverKind::GpuForm || d_.n_rows > (1 << 26) ||
        env_int("BW_RESIDENT", 1) == 0)
        return lists;
    const int slices_cap = std::min(RS_SETS_CAP, env_int("BW_GROUP_MIN", RS_SETS_CAP));
    pos.assign(col.size(), 0);
    // per row: the last part that met it, and its place among that part's
    // directions (own rows, then the halo)
    std::vector<int> met(d_.n_rows, -1);
    std::vector<uint16_t> place(d_.n_rows, 0);
    int stamp = -1;
    for (int i = 0; i < size(); i++)
    {
        const int n = nslices_[i], count = (n + hold - 1) / hold;
        if (n > slices_cap || count > PARTS_CAP || params[i].max_iter > ITER_CAP)
            continue;
        const size_t part0 = part.size(), halo0 = halo_row.size();
        int longest = 0, s = slice_base_[i];
        for (int k = 0; k < count; k++)
        {
            ResidentPart p = {};
            p.inst = i;
            p.slice0 = s;
            p.n_slices = std::min(hold, n - k * hold);
            p.sets = n;
            p.set0 = slice_base_[i];
            p.halo_off = (int)halo_row.size();
            p.parts = count;
            s += p.n_slices;
            const int r0 = p.slice0 * SLICE, r1 = s * SLICE;
            const size_t e0 = slice_off[p.slice0],
                         e1 = slice_off[s - 1] + (size_t)slice_w[s - 1] * SLICE;
            rows.clear();
            stamp++;
            for (int c = r0; c < r1; c++)
            {
                met[c] = stamp;
                place[c] = (uint16_t)(c - r0);
            }
            for (size_t e = e0; e < e1; e++)
            {
                const int c = col[e];
                if (met[c] != stamp)
                {
                    met[c] = stamp;
                    rows.push_back(c);
                }
            }
            p.halo_n = (int)rows.size();
            longest = std::max(longest, p.halo_n);
            if (longest > halo_cap(fp32))
                break;
            std::sort(rows.begin(), rows.end());
            for (size_t h = 0; h < rows.size(); h++)
                place[rows[h]] = (uint16_t)(hold * SLICE + h);
            for (size_t e = e0; e < e1; e++)
                pos[e] = place[col[e]];
            halo_row.insert(halo_row.end(), rows.begin(), rows.end());
            part.push_back(p);
        }
        if (longest > halo_cap(fp32))
        {
            part.resize(part0);
            halo_row.resize(halo0);
            continue;
        }
        rp.first[i] = (int)part0;
        rp.count[i] = count;
        rp.most = std::max(rp.most, count);
        rp.sets_max = std::max(rp.sets_max, n);
        rp.halo_max = std::max(rp.halo_max, (longest + 1) & ~1);
        for (size_t k = part0; k < part.size(); k++)
        {
            int extra = 0;
            for (int sl = part[k].slice0; sl < part[k].slice0 + part[k].n_slices; sl++)
                extra += std::max(0, slice_w[sl] - RS_SLOTS);
            rp.extra = std::max(rp.extra, extra);
        }
    }
    rp.parts = (int)part.size();
    return lists;
}

void Batch::build_resident(const ResidentLists &lists)
{
    const bool fp32 = kind_ == SolverKind::CG32;
    ResidentPlan &rp = resident_;
    if (rp.parts == 0)
        return;
    // one allocation for all arrays (each costs a fill and a wait), the ones
    // with contents first, uploaded together
    typedef unsigned long long u64;
    size_t bytes = 0;
    auto place = [&](size_t n) {
        const size_t at = bytes;
        bytes += (n + 255) & ~(size_t)255;
        return at;
    };
    auto size_of = [](const auto &v) { return v.size() * sizeof(v[0]); };
    const size_t rows = d_.n_rows, slices = d_.n_slices;
    const size_t part = place(size_of(lists.part)), halo = place(size_of(lists.halo_row)),
                 pos = place(size_of(lists.pos)), table = place(sizeof(ResidentBatch)),
                 contents = bytes;
    const size_t z = place(rows * 3 * (fp32 ? 1 : 2) * sizeof(u64)),
                 x = place(rows * 6 * sizeof(u64)), s_dq = place(slices * 2 * sizeof(u64)),
                 s_rz = place(slices * 4 * sizeof(u64)), s_res = place(slices * 6 * sizeof(u64)),
                 epoch = place(size() * sizeof(unsigned));
    const size_t ctl_bytes = sizeof(ResidentCtl) + (size_t)rp.parts * sizeof(int2);
    const size_t ctl = place(ctl_bytes);
    char *base = dalloc<char>(bytes);
    ResidentBatch &rb = rp.entry;
    rb.d = d_;
    rb.part = reinterpret_cast<ResidentPart *>(base + part);
    rb.halo_row = reinterpret_cast<int *>(base + halo);
    rb.pos = reinterpret_cast<uint16_t *>(base + pos);
    rb.z = reinterpret_cast<u64 *>(base + z);
    rb.x = reinterpret_cast<u64 *>(base + x);
    rb.s_dq = reinterpret_cast<u64 *>(base + s_dq);
    rb.s_rz = reinterpret_cast<u64 *>(base + s_rz);
    rb.s_res = reinterpret_cast<u64 *>(base + s_res);
    rb.epoch = reinterpret_cast<unsigned *>(base + epoch);
    std::vector<char> head(contents);
    auto put = [&](size_t at, const void *src, size_t n) {
        if (n)
            std::memcpy(head.data() + at, src, n);
    };
    put(part, lists.part.data(), size_of(lists.part));
    put(halo, lists.halo_row.data(), size_of(lists.halo_row));
    put(pos, lists.pos.data(), size_of(lists.pos));
    put(table, &rb, sizeof rb);
    check(hipMemcpy(base, head.data(), contents, hipMemcpyHostToDevice), "hipMemcpy H2D");
    if (opt_.shared_launches)
        return; // the server has the table and the tickets
    rp.table = reinterpret_cast<ResidentBatch *>(base + table);
    rp.ctl = base + ctl;
    check(hipHostMalloc((void **)&rp.host_ctl, ctl_bytes), "hipHostMalloc");
}

void Batch::free_resident()
{
    if (resident_.host_ctl)
        (void)hipHostFree(resident_.host_ctl);
    resident_.host_ctl = nullptr;
}

bool Batch::all_resident() const
{
    if (resident_.parts == 0 || resident_.given_up)
        return false;
    for (int c : resident_.count)
        if (c == 0)
            return false;
    return true;
}

// Solves that start on the FP64 matrix (after a stall in the step before) go by
// launches where those are faster: the one launch reads that matrix with a CU a
// part only.  us an iteration, one launch and launches (1 lane per row): 33 x 33
// 11.5 and 9.1, 65 x 65 11.9 and 10.0, 125 x 125 12.1 and 10.1, 210 x 210 (692
// slices) 17.4 and 16.3, 257 x 257 18.5 and 19.6, one part (21 x 21) 8.2 and 9.5;
// 2 of 97 x 97 (296 slices) 12.1 and 11.2, 5 of 65 x 65 (340) 11.6 and 11.2, 2 of
// 125 x 125 (496) 12.3 and 12.6; 8 of 33 x 33 11.3 and 11.9.  A batch whose other
// cloths go in the one launch keeps these there, beside them.
// A cloth alone that moves on to that matrix in mid-solve leaves the launch too
// (a drape's solve of 51,920 iterations: 604 ms in one launch, 538 by launches
// from the start, 514 so).
bool Batch::w64_size() const
{
    return kind_ == SolverKind::CG32 && size() < 8 && resident_.most > 1 &&
           d_.n_slices <= (size() == 1 ? 700 : 350);
}

bool Batch::w64_by_launches() const
{
    if (!w64_size())
        return false;
    for (char w : w64_next_)
        if (!w)
            return false;
    return true;
}

// One launch over the resident cloths, after the reset of their states on
// the batch's stream.  Cloths go in the order of the iterations that they
// took in the last solve, the most first (in the first solve: of their
// slices), since a launch lasts as long as its last cloth.  Returns false
// when the launch is not possible here or was given up (a wait ran out
// because other work kept the chip from holding a cloth's workgroups at
// once): then `again` has assembled the system a second time, every state is
// that of a solve's start, and the batch solves by launches from now on.
bool Batch::solve_resident(const std::function<void()> &again)
{
    const bool fp32 = kind_ == SolverKind::CG32;
    ResidentPlan &rp = resident_;
    const int extra = resident_extra(fp32, rp.sets_max, rp.halo_max, rp.extra);
    const size_t lds = resident_lds(fp32, rp.sets_max, rp.halo_max, extra);
    const int lpr = kind_ == SolverKind::RefPCG64 ? 0 : d_.spmv_lpr;
    if (rp.lpr != lpr)
    {
        rp.lpr = lpr;
        rp.capacity = resident_capacity(fp32, rp.lpr, lds);
    }
    if (rp.capacity < rp.most)
    {
        rp.given_up = true;
        return false;
    }
    std::vector<int> &order = lane_order_;
    order.clear();
    for (int i = 0; i < size(); i++)
        if (rp.count[i] > 0)
            order.push_back(i);
    const bool known = (int)pred_launches_.size() == size();
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return known ? pred_launches_[a] > pred_launches_[b] : nslices_[a] > nslices_[b];
    });
    ResidentCtl *ctl = reinterpret_cast<ResidentCtl *>(rp.host_ctl);
    *ctl = ResidentCtl{};
    int2 *ticket = reinterpret_cast<int2 *>(ctl + 1);
    for (int i : order)
        for (int k = 0; k < rp.count[i]; k++)
            *ticket++ = make_int2(0, rp.first[i] + k);
    ResidentLaunch a = {};
    a.table = rp.table;
    a.ctl = reinterpret_cast<ResidentCtl *>(rp.ctl);
    a.tickets = rp.parts;
    a.lpr = rp.lpr;
    a.sets_max = rp.sets_max;
    a.halo_max = rp.halo_max;
    a.extra = extra;
    resident_limits(a, *ctl, size() == 1 && w64_size());
    int aborted = 0;
    {
        const int grid = std::min(rp.parts, rp.capacity);
        ResidentSeats seats;
        if (rp.most > 1)
            seats.take(grid);
        check(hipMemcpyAsync(rp.ctl, rp.host_ctl,
                             sizeof(ResidentCtl) + (size_t)rp.parts * sizeof(int2),
                             hipMemcpyHostToDevice, stream_),
              "hipMemcpyAsync tickets");
        launch_resident(a, fp32, grid, stream_);
        check(hipGetLastError(), "resident launch");
        check(hipMemcpyAsync(rp.host_ctl, rp.ctl, sizeof(ResidentCtl), hipMemcpyDeviceToHost,
                             stream_),
              "hipMemcpyAsync control");
        check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
        aborted = ctl->aborted;
    }
    if (!aborted)
        return true;
    rp.given_up = true;
    again();
    launch_cg_restart(d_, stream_);
    return false;
}

void Batch::restart_step()
{
    resident_.given_up = true;
    launch_assemble_rows(d_, stream_);
    launch_cg_restart(d_, stream_);
    check(hipGetLastError(), "step launch");
}

} // namespace bw
