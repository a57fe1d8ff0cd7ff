// Which persistent launches of a device have to be put behind which (launch_persistent in recurrent.hip).  Bookkeeping
// alone, without HIP: a Stream is any handle that compares.
#pragma once

namespace flstm_hip {

// One per device, used under its owner's lock.  Only the last launch is remembered: every launch was put behind the one
// before it, so when the last one is over, all are.
template <typename Stream>
class LaunchGate {
public:
    // per_thread: the handle that names another stream in every thread
    explicit LaunchGate(Stream per_thread) : per_thread_(per_thread) {}

    // The last launch may still be running, and a launch to `stream` would not be in order behind it.
    bool must_wait(Stream stream) const { return in_flight_ && (stream != last_ || stream == per_thread_); }
    Stream last() const { return last_; }
    // The end of the last launch already has an event: a launch through the per-thread handle needs one from its own
    // thread, since no other thread can name that stream.
    bool recorded() const { return recorded_; }
    bool wants_event(Stream stream) const { return stream == per_thread_; }

    void launched(Stream stream, bool recorded) {
        last_ = stream;
        recorded_ = recorded;
        in_flight_ = true;
        ++launches_;
    }
    // To be taken before a stream is waited for and handed to waited() afterwards.
    unsigned long launches() const { return launches_; }
    // `stream` has been waited for.  A launch that another thread made meanwhile, to the same stream too, may have come
    // after that wait began: then nothing is known.  Nor is it known of which thread's stream a per-thread handle spoke.
    void waited(Stream stream, unsigned long launches) {
        if (stream == last_ && stream != per_thread_ && launches == launches_) in_flight_ = false;
    }

private:
    Stream per_thread_, last_{};
    bool in_flight_ = false, recorded_ = false;
    unsigned long launches_ = 0;
};

}  // namespace flstm_hip
