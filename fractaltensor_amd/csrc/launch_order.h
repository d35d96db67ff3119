// When kernels whose workgroups wait for each other may be launched as ordinary kernels, and what a launch has to be put
// behind (launch_resident in ftk_api.hip).  No HIP in here: what is asked of the runtime comes in as a parameter.
#pragma once

namespace ftk {

enum class StreamState { kIdle, kBusy, kCapturing, kGone };

// Of one device.  Runtime:
//   bool capturing(Stream)               the stream records a graph
//   StreamState state(Stream)            of a stream that got an ordinary launch
//   int put_behind(Stream s, Stream of)  s goes on when what `of` holds now has ended; 0 or an error
//   int wait_for_device()                0 or an error
template <typename Stream>
class LaunchOrder {
 public:
  // How the next launch on s goes.  every_thread: one handle that is another stream in every thread.
  template <typename Runtime>
  int next(Runtime&& rt, Stream s, bool every_thread, bool* cooperative) {
    const bool capturing = rt.capturing(s);
    // a graph may be replayed on any stream, and later ordinary launches would not know
    if (capturing || every_thread) cooperative_ = true;
    bool ordered = !capturing;   // nothing can be put in front of what is only recorded: it stays to be done
    if (ordered && pending_ && (last_ != s || every_thread)) {
      int rc = 0;
      switch (rt.state(last_)) {
        case StreamState::kIdle:
          pending_ = false;
          break;
        case StreamState::kBusy:
          rc = rt.put_behind(s, last_);
          cooperative_ = true;
          break;
        case StreamState::kCapturing:   // must not be asked (that would end its capture), and nothing can be put behind it now
          cooperative_ = true;
          ordered = false;
          break;
        case StreamState::kGone:        // its work may not be
          rc = rt.wait_for_device();
          pending_ = false;
          break;
      }
      if (rc) return rc;
    }
    if (!cooperative_) {
      pending_ = true;
      last_ = s;
    } else if (ordered) {
      pending_ = false;   // cooperative launches run in turn: all later ones follow this one
    }
    *cooperative = cooperative_;
    return 0;
  }

  // Whether a launch on s is going to be cooperative, as far as can be told without making it: the first one on a second stream
  // may still turn out to be.
  template <typename Runtime>
  bool cooperative(Runtime&& rt, Stream s, bool every_thread) const {
    return cooperative_ || every_thread || rt.capturing(s);
  }

 private:
  bool cooperative_ = false;   // from the second stream on
  bool pending_ = false;       // ordinary launches on last_ may still run, and no cooperative launch has been put behind them
  Stream last_{};
};

}  // namespace ftk
