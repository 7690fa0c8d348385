// Mutual exclusion of the calls that run grid-synchronizing kernels on a device.
#pragma once

#include <fcntl.h>
#include <sys/file.h>
#include <sys/stat.h>
#include <unistd.h>

#include <cerrno>
#include <chrono>
#include <mutex>
#include <string>

namespace snhip {

// A grid of such a kernel fills the device, and two of them, each with part of its
// workgroups resident, would wait for each other. One call at a time holds the
// device's gate, from before its launch until its kernel has finished: among the
// threads of a process by mutexes, among processes by flock on two files. Who waits
// holds the turnstile (next_), so that a caller in a loop cannot pass through again
// before it. A process that ends, however it ends, gives its files' locks back. On
// an idle gate entering and leaving takes less than a microsecond.
class DeviceGate {
public:
    explicit DeviceGate(const std::string& path) : path_(path) {}
    ~DeviceGate() {
        if (fnext_ >= 0) close(fnext_);
        if (fhold_ >= 0) close(fhold_);
    }
    DeviceGate(const DeviceGate&) = delete;
    DeviceGate& operator=(const DeviceGate&) = delete;

    // Waits for the gate. False, and not held, if other processes cannot be kept out:
    // the files cannot be opened, or a holder has not let go for `limit` seconds (it is
    // stopped, or hangs; the next calls then do not wait until it has).
    bool enter(double limit) {
        next_.lock();
        hold_.lock();
        const bool all = enter_files(stuck_ ? 0.0 : limit);
        if (!all) hold_.unlock();
        next_.unlock();
        return all;
    }
    void leave() {
        (void)flock(fhold_, LOCK_UN);
        hold_.unlock();
    }

private:
    std::mutex next_, hold_;
    const std::string path_;
    bool opened_ = false, stuck_ = false;   // under hold_
    int fnext_ = -1, fhold_ = -1;

    // Any user of the device may lock the files: flock needs no write access.
    static int open_lock(const std::string& p) {
        const int flags = O_RDONLY | O_CLOEXEC | O_NOFOLLOW | O_NONBLOCK;
        int fd = open(p.c_str(), flags);
        if (fd < 0 && errno == ENOENT) {
            fd = open(p.c_str(), flags | O_CREAT | O_EXCL, 0444);
            if (fd >= 0) (void)fchmod(fd, 0444);                       // whatever the umask
            else if (errno == EEXIST) fd = open(p.c_str(), flags);     // another process was first
        }
        struct stat st;
        if (fd >= 0 && (fstat(fd, &st) != 0 || !S_ISREG(st.st_mode))) {
            close(fd);
            fd = -1;
        }
        return fd;
    }
    static bool lock_by(int fd, std::chrono::steady_clock::time_point end) {
        while (flock(fd, LOCK_EX | LOCK_NB) != 0) {
            if (errno != EWOULDBLOCK && errno != EINTR) return false;
            if (std::chrono::steady_clock::now() >= end) return false;
            usleep(20);
        }
        return true;
    }
    bool enter_files(double limit) {
        if (!opened_) {
            opened_ = true;
            fnext_ = open_lock(path_ + ".next");
            fhold_ = open_lock(path_);
        }
        if (fnext_ < 0 || fhold_ < 0) return false;
        const auto end = std::chrono::steady_clock::now() +
                         std::chrono::duration_cast<std::chrono::steady_clock::duration>(std::chrono::duration<double>(limit));
        stuck_ = !lock_by(fnext_, end);
        if (stuck_) return false;
        stuck_ = !lock_by(fhold_, end);
        (void)flock(fnext_, LOCK_UN);
        return !stuck_;
    }
};

}  // namespace snhip
