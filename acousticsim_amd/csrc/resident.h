// One-launch tolerance solves (resident.hip): the device layout of a batch's
// cloths as parts, one workgroup each, and the launcher.
#pragma once
#include "device.h"

namespace bw
{

// Slices (64 rows, one wavefront each) of a part, by the solver's precision,
// and matrix slots of a row that its registers keep.  8 in the mixed form:
// with 4, a cloth has twice the parts, and the exchange costs more than the
// shorter chains save (125 x 125 5.9 us an iteration against 5.4, 257 x 257
// 12.2 against 9.3; only some 65 x 65 cloths gain).  4 in FP64, whose blocks
// fill twice the registers.
constexpr int RS_WAVES32 = 8, RS_WAVES64 = 4;
constexpr int resident_slices(bool fp32) { return fp32 ? RS_WAVES32 : RS_WAVES64; }
constexpr int RS_SLOTS = 13;
// slices of the largest cloth that one launch solves
constexpr int RS_SETS_CAP = 1088;
// LDS of a part's workgroup at most, and of one more slot of a slice there
// (nine values and a position a row)
constexpr size_t RS_LDS_MAX = 160 * 1024 - 1024;
constexpr size_t resident_slot_bytes(bool fp32)
{
    return SLICE * (9 * (fp32 ? sizeof(float) : sizeof(double)) + sizeof(unsigned));
}
// longest halo of a part (rows), by the solver's precision: with the sums of
// the largest cloth (resident_plan.cpp) it fits the CU's 160 KiB of LDS
constexpr int RS_HALO32 = 2688, RS_HALO64 = 2176;
// Slices slice0 .. slice0 + n_slices - 1 of a cloth, solved by one workgroup
// with the cloth's other parts. halo_off / halo_n: the rows of other parts
// that its rows read (ResidentBatch::halo_row).
struct ResidentPart
{
    int inst, slice0, n_slices;
    int sets;       // slices of the whole cloth (partial sums to add)
    int set0;       // the cloth's first slice
    int halo_off, halo_n;
    int parts;      // workgroups of the cloth
};

// A batch as the kernel sees it (a device table of these: a launch may run
// cloths of several batches)
struct ResidentBatch
{
    DeviceBatch d;
    const ResidentPart *part;
    const int *halo_row;
    // per ELL entry (indexed like col): its column's position in the part's
    // direction array, own rows first, then the halo
    const uint16_t *pos;
    // exchange words, {tag, 32 bits of a value}: z of every row (3 values),
    // the solution of every row (3 doubles), and the partial sums of every
    // slice: d.q (1 double), r.z and r.r (2), those of a true residual (3)
    unsigned long long *z, *x, *s_dq, *s_rz, *s_res;
    unsigned *epoch; // per cloth: the last tag used
};

// Launch control, at the head of the ticket buffer
struct ResidentCtl
{
    int next;     // next ticket
    int aborted;  // 1: a wait ran out; the launch's cloths are not solved
    int progress; // moves on while any of the launch's cloths does
    int pad;
    // of the 100 MHz clock, without a wait's end or progress of any cloth
    unsigned long long wait_ticks;
};

struct ResidentLaunch
{
    const ResidentBatch *table; // device
    ResidentCtl *ctl;           // device; the tickets (int2 {batch, part}) follow it
    int tickets;
    // the rounding it follows: of the SpMV variant with 1, 2 or 4 lanes per
    // row, or of the reference-semantics solver (0)
    int lpr;
    int sets_max, halo_max;     // over the launch's parts (halo_max even)
    int extra;                  // slots of slices past RS_SLOTS that a part keeps in LDS
    // tests: abort a cloth after this many iterations (0: never); < 0: a cloth
    // that moves on to the FP64 matrix leaves the launch, for the launches to
    // finish (one cloth only)
    int give_up;
    // iterations of a cloth after which its solve pauses until the next launch
    // (0: never); only with one lane per row
    int pause;
};

// The workgroups of a cloth of several parts wait for one another, so two
// launches that each held part of the chip would both wait.  Launches with such
// clothes take a seat a workgroup, from the launch until it has ended, and
// together no more than the device has CUs, so that each has all of its
// workgroups running whatever CUs the others' are on; a launch whose clothes
// have one part each waits for nothing and takes none.  First come, first
// served; a launch with more workgroups than CUs takes them all.
class ResidentSeats
{
public:
    ResidentSeats() = default;
    ResidentSeats(const ResidentSeats &) = delete;
    ResidentSeats &operator=(const ResidentSeats &) = delete;
    ~ResidentSeats() { give(); }
    void take(int n); // on the current device; waits
    void give();      // all that were taken

private:
    struct Device;
    Device *of_ = nullptr;
    int n_ = 0;
};
// slots of slices past RS_SLOTS that a part can keep in LDS, of `wanted`
int resident_extra(bool fp32, int sets_max, int halo_max, int wanted);
// when a launch is given up: after a wait of 2 s in which none of its cloths
// got on (BW_RESIDENT_WAIT_MS), or at BW_RESIDENT_GIVE_UP iterations of a
// cloth (tests)
// (w64_leaves: and a cloth leaves it when it moves on to the FP64 matrix)
void resident_limits(ResidentLaunch &a, ResidentCtl &ctl, bool w64_leaves = false);
// dynamic LDS bytes of a launch
size_t resident_lds(bool fp32, int sets_max, int halo_max, int extra);
// workgroups of the launch that are resident at once on the current device
// (0 when the kernel cannot run with that LDS)
int resident_capacity(bool fp32, int lpr, size_t lds, bool pause = false);
void launch_resident(const ResidentLaunch &a, bool fp32, int grid, hipStream_t s);
// solver states of a solve that is started again (after an aborted launch):
// the solve start, with the history that k_cg_reset had given it
void launch_cg_restart(const DeviceBatch &d, hipStream_t s);

} // namespace bw
