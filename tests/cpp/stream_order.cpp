// Runs StreamOrderT over a device of names: a stream is the set of operations
// that have finished before whatever it is given next. Reads one command per
// line and prints a line per operation: its number and whether every earlier
// operation of the handle has finished before it starts.
//   bind S     the handle is bound to stream S (P: the per-thread stream)
//   thread N   the calls come from thread N
//   async      an operation of the handle that returns before it is done
//   quiet      one that does not mark
//   capture S  S is being captured from here on; endcapture S ends it (a call on
//              it prints nothing: it runs when the capture is replayed)
//   free       the handle's last wait: prints whether all operations are done
#include <cstdint>
#include <iostream>
#include <map>
#include <string>

#include "streamorder.h"

struct Dev {
    std::map<unsigned long long, uint64_t> streams;   // by number
    std::map<std::string, unsigned long long> ids;
    std::map<std::string, bool> cap;
    std::string thread;
    uint64_t host = 0;
    unsigned long long next = 0;
};
static Dev dev;
static unsigned long long number(const std::string& s) {
    unsigned long long& n = dev.ids[s == "P" ? s + dev.thread : s];
    return n ? n : n = ++dev.next;
}

struct Rt {
    using Stream = std::string;
    using Event = uint64_t*;
    using Error = int;
    static constexpr int ok = 0;
    static unsigned long long id(Stream s) { return number(s); }
    static int capturing(Stream s, bool* c) { *c = dev.cap[s]; return ok; }
    static int create(Event* e) { *e = new uint64_t(0); return ok; }
    static void destroy(Event e) { delete e; }
    static int record(Event e, Stream s) { if (dev.cap[s]) return 1; *e = dev.streams[number(s)]; return ok; }
    static int wait(Stream s, Event e) { if (dev.cap[s]) return 2; dev.streams[number(s)] |= *e; return ok; }
    static int host_wait(Event e) { dev.host |= *e; return ok; }
};

int main() {
    snhip::StreamOrderT<Rt> order;
    std::string cmd, cur;
    uint64_t all = 0;
    int n = 0;
    auto check = [](int e) { if (e) std::cout << "error " << e << "\n"; };
    while (std::cin >> cmd) {
        if (cmd == "bind") {
            std::cin >> cur;
        } else if (cmd == "thread") {
            std::cin >> dev.thread;
        } else if (cmd == "capture" || cmd == "endcapture") {
            std::string s;
            std::cin >> s;
            dev.cap[s] = cmd == "capture";
        } else if (cmd == "free") {
            check(order.drain());
            const uint64_t done = dev.host | dev.streams[number(cur)];
            std::cout << "free " << ((done & all) == all) << "\n";
        } else {
            check(order.follow(cur));
            if (!dev.cap[cur]) {
                const uint64_t done = dev.host | dev.streams[number(cur)];
                std::cout << n << " " << ((done & all) == all) << "\n";
                all |= 1ull << n;
                dev.streams[number(cur)] |= 1ull << n;
                ++n;
            }
            if (cmd == "async") check(order.mark(cur));
        }
    }
}
