// Runs DeviceGate in threads and processes. dev_gate MODE PATH ...
//   excl PATH THREADS ROUNDS COUNTER   every thread passes the gate ROUNDS times, and
//       inside it reads, waits and writes back the number in COUNTER plus one
//   loop PATH SECONDS                  passes it without a pause; prints how often
//   hold PATH SECONDS                  enters, prints "in", sleeps holding it
//   try PATH LIMIT [N PAUSE]           tries to enter once (N times, PAUSE seconds apart),
//                                      prints whether it did and how long it took
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "devgate.h"

static double now() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

int main(int argc, char** argv) {
    const std::string mode = argv[1];
    snhip::DeviceGate gate(argv[2]);
    if (mode == "excl") {
        const int threads = atoi(argv[3]), rounds = atoi(argv[4]);
        std::vector<std::thread> ts;
        for (int i = 0; i < threads; ++i)
            ts.emplace_back([&] {
                for (int r = 0; r < rounds; ++r) {
                    if (!gate.enter(60)) exit(3);
                    long v = 0;
                    FILE* f = fopen(argv[5], "r");
                    if (!f || fscanf(f, "%ld", &v) != 1) exit(4);
                    fclose(f);
                    usleep(50);
                    f = fopen(argv[5], "w");
                    fprintf(f, "%ld\n", v + 1);
                    fclose(f);
                    gate.leave();
                }
            });
        for (auto& t : ts) t.join();
    } else if (mode == "loop") {
        const double end = now() + atof(argv[3]);
        long n = 0;
        for (; now() < end; ++n) {
            if (!gate.enter(60)) return 3;
            usleep(300);
            gate.leave();
        }
        printf("%ld\n", n);
    } else if (mode == "hold") {
        if (!gate.enter(60)) return 3;
        printf("in\n");
        fflush(stdout);
        usleep((useconds_t)(atof(argv[3]) * 1e6));
        gate.leave();
    } else if (mode == "try") {
        for (int i = 0; i < (argc > 4 ? atoi(argv[4]) : 1); ++i) {
            if (i) usleep((useconds_t)(atof(argv[5]) * 1e6));
            const double t = now();
            const bool in = gate.enter(atof(argv[3]));
            printf("%d %.3f\n", in, now() - t);
            fflush(stdout);
            if (in) gate.leave();
        }
    }
    return 0;
}
