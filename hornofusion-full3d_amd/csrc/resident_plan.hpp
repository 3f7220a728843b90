// resident_plan.hpp -- host side of the resident solvers: which batches
// they take, the teams, and the launch's device tables.
#pragma once
#include <chrono>
#include <memory>
#include <vector>

#include "batch.hpp"
#include "resident.hpp"

namespace eafp {

// What a resident kernel of one solver can hold and about what its
// iterations cost; the plan picks the team size by it.
struct ResLimits {
    int max_slots;                            // slots per thread
    int (*slots)(int nz, int rows);           // slots per thread for `rows` z-rows, 0: none fits
    size_t (*lds)(int nz, int rows, int lds_rows, int halo_rows);
    float sync_us[9];                         // two team sums and the exchange, T = 1, 2, 4 .. 256
    float slot_us;                            // one slot's iteration
};

struct ResPlan {
    bool ok = false;
    int nsys = 0;
    int T = 0, nteam = 0, blocks = 0;         // T = 0: teams of different sizes
    int members = 0;                          // work-groups that wait for each other (0: teams of one)
    int slots = 0;                            // largest over the items
    size_t lds = 0;
    int max_items = 0;                        // longest team list
    float est_us = 0.f;                       // model: one iteration of every system
    std::vector<ResItem> items;               // team by team
    std::vector<int> team_begin;
    std::vector<ResTeam> teams;               // with T = 0
    std::vector<int2> member;
    int nslot = 0;                            // slots of all teams
    long xlen = 0;                            // elements of the exchange buffer
    // the CUs it takes: teams of one do not wait for each other, but others'
    // launches would wait for them, longer than the gate does where lists are long
    int places() const { return members > 0 ? members : nteam; }
};

// The plan for a batch, or !ok when a system fits no team.  `xpitch`: the
// exchange buffer's elements per z-row.
ResPlan plan_resident(const std::vector<SysGeom>& g, const ResLimits& lim, int (*xpitch)(int nz));

// Work-groups of resident launches in flight on this process's GPUs: a launch
// takes its number before it is queued and gives it back when it has ended,
// waiting in turn when the CUs are taken, so that two launches never hold
// half of the CUs each.
class ResidentGate {
  public:
    explicit ResidentGate(int blocks);
    ~ResidentGate();
    ResidentGate(const ResidentGate&) = delete;
    ResidentGate& operator=(const ResidentGate&) = delete;

  private:
    int dev_, n_;
};

// Launches that the autotuner times of a resident form; it keeps the least time,
// so that one launch held up does not send a batch to the streaming kernels.
constexpr int RES_TIMED = 5;

// A plan's tables on the device: some kilobytes, as rows are exchanged through an
// array that the solver's resident kernel does not use otherwise, and given
// back should the solver run out of memory later.
struct ResDevice {
    ResPlan plan;
    DevBuf<ResItem> items;
    DevBuf<int> team_begin;
    DevBuf<ResTeam> teams;
    DevBuf<int2> member;
    DevBuf<u64> slots;
    DevBuf<unsigned> gate;
    unsigned tag = 1;             // first tag of the next launch
    // A launch that did not get its CUs has cost time (resident.hpp), and the
    // batch streams until RES_RETRY times as long has passed: with the CUs held
    // by others for good, a hundredth of the time is lost, and after a single
    // collision the solves are on chip again.
    std::chrono::steady_clock::time_point retry{};
    bool usable() const { return std::chrono::steady_clock::now() >= retry; }
    void gave_up(std::chrono::steady_clock::time_point since);
    long long launches = 0, given_up = 0, aside = 0;   // of resident launches, given up, systems set aside
    int absent = 0;               // work-groups that a launch waits for and that never come (tests)
    int init(ResPlan&& p, hipStream_t stream);
    ResLaunch launch() const;
    // `out` stays empty, and the batch streams, where the plan is not ok or the
    // device's memory does not hold its tables
    static int create(ResPlan&& p, std::unique_ptr<ResDevice>& out, hipStream_t stream);
    // gate open and `tag` set for the next launch, which uses at most `tags` of them
    int arm(long tags, hipStream_t stream);
    // the first of `tags` tags, for a kernel that opens the gate itself
    int take_tags(long tags, hipStream_t stream, unsigned* first);
};

__global__ void k_res_arm(unsigned* gate, unsigned tag);

}  // namespace eafp
