// mdn_team_plan.h -- the host side of the persistent minimizer's teams (mdn_team.h): how many
// workgroups a network gets, how a batch's workgroups are shared out, and how many workgroups that
// wait for each other may be in flight on a device. No HIP: also compiled into a CPU check.
//
// Workgroups of a team wait for each other, and each of them fills a CU, so a team only gets on once
// all of it is resident. A cooperative launch guarantees that, but it goes through a queue of its own:
// teams of several contexts then run one after the other, and once that queue exists everything else
// that a process runs on four streams is slowed down (7,500 beads by four threads, no team among
// them: 1,270 us per minimization without the queue, 3,660 with it; 550 beads by teams: 1,195).
// Teams are therefore launched like any other kernel, and TeamRoom keeps those in flight to what
// fits: whoever finds no room left takes the form that waits for nobody (the four-kernel slots, a
// batch of single workgroups), with the same result.
#pragma once

#include <algorithm>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace mdn {

constexpr int TEAM_MAX = 32;   // workgroups of a team: the CUs of an XCD

// One team: its workgroups and the system it owns (sys < 0: a single workgroup that pulls systems
// from the queue).
struct TeamInfo {
    int size, sys;
};
struct TeamSlot {   // per workgroup: its team (< 0: none) and its place in it
    int team, member;
};

// Workgroups of teams that are resident together for certain: those of one XCD. Which XCD a launch's
// first workgroup runs on depends on its hardware queue, so any two teams may meet on the same one.
// A partition holds whole XCDs; a device that shows fewer CUs than one has the CUs it shows.
inline int team_room(int n_cu) { return std::max(1, std::min(TEAM_MAX, n_cu)); }

// The workgroups of teams in flight on one device. A call may wait for its share for a while; as long
// as one does, those that don't wait get none, so that it is not passed over for ever.
struct TeamRoom {
    std::mutex mu;
    std::condition_variable freed;
    int used = 0, waiting = 0;
    bool take(int n, int room, std::chrono::microseconds wait) {
        std::unique_lock<std::mutex> lk(mu);
        const auto fits = [&] { return n <= room - used; };
        if (wait.count() > 0) {
            waiting++;
            const bool ok = freed.wait_for(lk, wait, fits);
            waiting--;
            if (!ok) return false;
        } else if (waiting > 0 || !fits()) {
            return false;
        }
        used += n;
        return true;
    }
    void give(int n) {
        {
            std::lock_guard<std::mutex> lk(mu);
            used -= n;
        }
        freed.notify_all();
    }
};
// A batch waits up to this long for its room: about what it loses by single workgroups (24 networks
// alone 2.0 ms by teams, 6.0 by single workgroups; by two and three threads 1.8 and 2.2 to 3.1 ms a batch
// where those that find the room taken go on at once, 1.4 and 1.6 with the wait).
constexpr std::chrono::microseconds TEAM_ROOM_WAIT{5000};
// A call's share of a room (null: none), given back by give() or at the end of the scope.
struct TeamHold {
    TeamRoom* room;
    int n = 0;
    explicit TeamHold(TeamRoom* r) : room(r) {}
    TeamHold(const TeamHold&) = delete;
    TeamHold& operator=(const TeamHold&) = delete;
    ~TeamHold() { give(); }
    bool take(int k, int size, std::chrono::microseconds wait = std::chrono::microseconds(0)) {
        if (!room || !room->take(k, size, wait)) return false;
        n = k;
        return true;
    }
    void give() {
        if (n) room->give(n);
        n = 0;
    }
};

// Work per workgroup below which another workgroup does not pay: batches of 8, 16 and 48 networks
// of up to 12,000 beads take 2.3, 2.6 and 4.4 ms with 256, 2.8, 3.0 and 4.7 ms with 1024, 3.5, 3.8
// and 5.7 ms with 2048.
constexpr long TEAM_SHARE = 256;
// A single network's work, in which a pair counts less than in a batch (its two chains run side by
// side): TEAM_ONE_SHARE of it per workgroup up to 16 workgroups, 24 from TEAM_WIDE on (below, their
// dearer barriers count more than the work they share) and from TEAM_ONE_MAX on the four-kernel
// slots over the whole chip. FP64 / mixed, ms per 80 iterations without the rebuild:
//   550 beads, work 1,200: 6, 8, 10 and 16 workgroups 1.30, 1.32, 1.36, 1.39 / 1.41, 1.41, 1.41, 1.44
//   4,200 in a sphere, 8,800: 16 and 24 workgroups 1.73, 1.67 / 1.60, 1.72
//   7,350 in a sphere, 13,900: 16, 24, 32, slots 2.13, 1.87, 1.91, 2.02 / 1.95, 1.87, 1.82, 2.17
//   3,150 in a cube, 14,200: 2.19, 1.93, 1.94, 2.12 / 2.01, 1.84, 1.90, 2.17
//   9,450 in a sphere, 19,100: 2.50, 2.11, 2.06, 2.04 / 2.23, 1.94, 2.01, 2.10
//   4,830 in a cube, 21,200: 2.69, 2.36, 2.22, 2.17 / 2.28, 2.18, 2.07, 2.17
// The one line for both precisions is FP64's: the mixed path would gain up to 8 % from teams between
// TEAM_ONE_MAX and a work of about 21,000, and 3 % from 32 workgroups at 13,900.
constexpr long TEAM_ONE_SHARE = 160, TEAM_WIDE = 9000, TEAM_ONE_MAX = 17500;
// Workgroups of the persistent minimizer for a single network; 0: the four-kernel slots.
inline int team_size_one(long work, int room) {
    if (work > TEAM_ONE_MAX) return 0;
    const long k = work > TEAM_WIDE ? 24 : std::min<long>(16, (work + TEAM_ONE_SHARE - 1) / TEAM_ONE_SHARE);
    return (int)std::min<long>(k, room);
}

// A batch's workgroups: which team each is in, and which system each team has. Large systems get
// teams of their own, sized to their share of the work; the others are pulled from a queue,
// largest first, by single workgroups. Workgroups b and b + 8 run on one XCD, and a team's
// workgroups are taken from one XCD. most: the most workgroups a team may have (1: a batch that
// waits for nobody).
struct TeamPlan {
    std::vector<TeamSlot> slot;
    std::vector<TeamInfo> team;
    std::vector<int> order;   // the queue
    int teamed = 0;           // workgroups of teams of more than one: they wait for each other
};
inline TeamPlan plan_teams(const std::vector<long>& cost, int groups, int most) {
    const int n = (int)cost.size(), NX = 8;
    TeamPlan P;
    std::vector<int> room(NX, 0);
    for (int b = 0; b < groups; b++) room[b % NX]++;
    most = std::min(std::min(TEAM_MAX, most), room[0]);
    long total = 0;
    for (long c : cost) total += c;
    std::vector<int> k(n, 1), by(n);
    for (int i = 0; i < n; i++) by[i] = i;
    std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return cost[a] > cost[b]; });
    // the share of work per workgroup, raised until the teams and the queue's workgroups fit
    for (double share = std::max<double>(TEAM_SHARE, (double)total / groups);; share *= 1.1) {
        int used = 0, small = 0;
        double rest = 0;
        for (int i = 0; i < n; i++) {
            k[i] = (int)std::max(1.0, std::min<double>(most, std::ceil(cost[i] / share)));
            if (k[i] > 1) used += k[i];
            else { small++; rest += cost[i]; }
        }
        if (used + std::min<double>(small, std::ceil(rest / share)) <= groups) break;
    }
    P.slot.assign(groups, TeamSlot{-1, 0});
    std::vector<int> taken(NX, 0);
    auto place = [&](int want, int sys) {   // a team of `want` workgroups on the XCD with the most room
        int x = 0;
        for (int q = 1; q < NX; q++)
            if (room[q] - taken[q] > room[x] - taken[x]) x = q;
        const int size = std::min(want, room[x] - taken[x]);
        if (size <= 0) return false;
        for (int m = 0; m < size; m++) P.slot[x + NX * (taken[x] + m)] = TeamSlot{(int)P.team.size(), m};
        taken[x] += size;
        P.team.push_back(TeamInfo{size, sys});
        if (size > 1) P.teamed += size;
        return true;
    };
    for (int i : by)
        if (k[i] == 1 || !place(k[i], i)) P.order.push_back(i);
    for (size_t j = 0; j < P.order.size(); j++)
        if (!place(1, -1)) break;
    return P;
}

}  // namespace mdn
