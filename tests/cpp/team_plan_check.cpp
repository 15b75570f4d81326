// The host side of the persistent minimizer's teams, checked on the CPU: sizes on devices with fewer
// CUs, the plan of a batch, and the room for teams under threads.
#include "../../picgo_amd/csrc/mdn_team_plan.h"

#include <atomic>
#include <cstdio>
#include <random>
#include <thread>

using namespace mdn;

static int bad = 0;
#define EXPECT(c) \
    do { if (!(c)) { bad++; std::printf("line %d: %s\n", __LINE__, #c); } } while (0)

int main() {
    // a single network's team fits the CUs that are there, on the chip and its partitions
    for (int n_cu : {1, 2, 5, 16, 32, 64, 128, 256, 304})
        for (long work : {1L, 159L, 161L, 1200L, 2560L, 9000L, 9001L, 17500L, 17501L, 1000000L}) {
            const int k = team_size_one(work, team_room(n_cu));
            EXPECT(k >= 0 && k <= n_cu && k <= TEAM_MAX && (work > TEAM_ONE_MAX) == (k == 0));
            if (n_cu >= 32) EXPECT(work > TEAM_ONE_MAX || work <= TEAM_WIDE || k == 24);
        }
    // a batch: every system has exactly one place, every team is whole, on one XCD, within the XCD's
    // CUs; with most = 1 nobody waits for anybody
    std::mt19937 g(3);
    for (int t = 0; t < 400; t++) {
        const int n = 1 + (int)(g() % 300), groups = 1 + (int)(g() % 256), most = t % 3 ? TEAM_MAX : 1;
        std::vector<long> cost(n);
        for (long& c : cost) c = 1 + (long)(g() % (t % 2 ? 3000 : 60000));
        const TeamPlan P = plan_teams(cost, groups, most);
        std::vector<int> seen(n, 0), members(P.team.size(), 0), xcd(P.team.size(), -1);
        int workers = 0, teamed = 0;
        EXPECT((int)P.slot.size() == groups);
        for (int b = 0; b < groups; b++) {
            const TeamSlot s = P.slot[b];
            if (s.team < 0) continue;
            EXPECT(s.team < (int)P.team.size());
            EXPECT(s.member >= 0 && s.member < P.team[s.team].size);
            members[s.team]++;
            EXPECT(xcd[s.team] < 0 || xcd[s.team] == b % 8);
            xcd[s.team] = b % 8;
        }
        for (size_t k = 0; k < P.team.size(); k++) {
            EXPECT(members[k] == P.team[k].size && P.team[k].size <= most);
            if (P.team[k].sys >= 0) seen[P.team[k].sys]++;
            else { workers++; EXPECT(P.team[k].size == 1); }
            if (P.team[k].size > 1) teamed += P.team[k].size;
        }
        for (int i : P.order) seen[i]++;
        for (int s : seen) EXPECT(s == 1);
        EXPECT(P.order.empty() || workers > 0);
        EXPECT(teamed == P.teamed && (most > 1 || P.teamed == 0));
    }
    // the room: what is in flight never passes it, all of it comes back, and a hold gives back at
    // the end of its scope, once
    TeamRoom room;
    std::atomic<int> now{0}, most{0}, got{0};
    std::vector<std::thread> th;
    for (int k = 0; k < 8; k++)
        th.emplace_back([&, k] {
            for (int i = 0; i < 20000; i++) {
                const int want = 1 + (k * 7 + i) % 32;
                TeamHold h(&room);
                if (!h.take(want, 32, std::chrono::microseconds(k < 2 ? 2000 : 0))) continue;
                got++;
                const int in = now += want;
                int m = most;
                while (in > m && !most.compare_exchange_weak(m, in)) {}
                now -= want;
                if (i % 2) h.give();
            }
        });
    for (auto& t : th) t.join();
    EXPECT(most <= 32 && got > 0 && room.used == 0);
    TeamHold none(nullptr), all(&room), late(&room);
    EXPECT(!none.take(1, 32) && all.take(32, 32) && !late.take(1, 32));
    all.give();
    EXPECT(late.take(1, 32) && room.used == 1);
    // whoever waits gets the room when it is given back, and not before; others don't pass it
    late.give();
    EXPECT(all.take(32, 32));
    const auto t0 = std::chrono::steady_clock::now();
    EXPECT(!late.take(32, 32, std::chrono::microseconds(3000)));
    EXPECT(std::chrono::steady_clock::now() - t0 >= std::chrono::microseconds(3000) && room.waiting == 0);
    std::thread w([&] { TeamHold h(&room); EXPECT(h.take(32, 32, std::chrono::seconds(20))); });
    for (bool seen = false; !seen;) {
        std::lock_guard<std::mutex> lk(room.mu);
        seen = room.waiting == 1;
    }
    all.n = 31;
    all.give();
    EXPECT(!late.take(1, 32));
    room.give(1);
    w.join();
    EXPECT(room.used == 0 && late.take(1, 32));
    std::printf("%d wrong\n", bad);
    return bad != 0;
}
