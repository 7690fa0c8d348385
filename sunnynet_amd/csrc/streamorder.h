// Order of one handle's calls across the streams they run on.
#pragma once

namespace snhip {

// Calls of one handle are in order also across changes of the caller's stream:
// each call that returns before its work is done marks the work's end on the
// stream it ran on (mark), and every call before the next mark on any other stream
// waits for it first (follow), however many there are. Streams are told apart by
// Rt's number for them and not by their handle: the per-thread stream has one handle
// in every thread. Rt supplies streams and events, so that the rule runs without a
// device too.
template <class Rt>
class StreamOrderT {
public:
    using Stream = typename Rt::Stream;
    using Error = typename Rt::Error;

    ~StreamOrderT() { if (ev_) Rt::destroy(ev_); }

    // (not while st is being captured: nothing has run there, and the earlier
    // mark still stands)
    Error mark(Stream st) {
        bool capturing = false;
        Error e = Rt::capturing(st, &capturing);
        if (e != Rt::ok || capturing) return e;
        if (!ev_ && (e = Rt::create(&ev_)) != Rt::ok) return e;
        if ((e = Rt::record(ev_, st)) != Rt::ok) return e;
        set_ = true;
        at_ = Rt::id(st);
        return Rt::ok;
    }
    // (A stream under capture cannot wait for an event from outside the capture:
    // the host waits instead.)
    Error follow(Stream st) {
        if (!set_ || Rt::id(st) == at_) return Rt::ok;
        bool capturing = false;
        const Error e = Rt::capturing(st, &capturing);
        if (e != Rt::ok) return e;
        return capturing ? Rt::host_wait(ev_) : Rt::wait(st, ev_);
    }
    // The host waits for the mark.
    Error drain() { return set_ ? Rt::host_wait(ev_) : Rt::ok; }

private:
    typename Rt::Event ev_{};
    bool set_ = false;
    unsigned long long at_ = 0;
};

}  // namespace snhip
