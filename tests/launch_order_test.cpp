// Scenarios for LaunchOrder (fractaltensor_amd/csrc/launch_order.h) against a runtime that only keeps a list of what it was
// asked for.  Prints the scenario that fails and ends with 1.
#include <cstdio>
#include <map>
#include <string>

#include "../fractaltensor_amd/csrc/launch_order.h"

using ftk::StreamState;

struct Fake {
  std::map<int, StreamState> streams;
  std::string log;   // what it was asked to do: "2>1 " stream 2 put behind stream 1, "wait "
  bool capturing(int s) { return streams[s] == StreamState::kCapturing; }
  StreamState state(int s) { return streams[s]; }
  int put_behind(int s, int of) {
    log += std::to_string(s) + ">" + std::to_string(of) + " ";
    return 0;
  }
  int wait_for_device() {
    log += "wait ";
    return 0;
  }
};

struct Device {
  Fake rt;
  ftk::LaunchOrder<int> order;
  // "o": ordinary, "c": cooperative, behind what the runtime was asked for
  std::string launch(int s, bool every_thread = false) {
    bool cooperative = false;
    rt.log.clear();
    if (order.next(rt, s, every_thread, &cooperative)) return "error";
    return rt.log + (cooperative ? "c" : "o");
  }
  // what it says the next one will be, without asking for anything else
  std::string ahead(int s, bool every_thread = false) {
    rt.log.clear();
    const bool cooperative = order.cooperative(rt, s, every_thread);
    return rt.log + (cooperative ? "c" : "o");
  }
};

static int failures = 0;
static void expect(const char* what, const std::string& got, const char* want) {
  if (got == want) return;
  std::printf("%s: '%s', expected '%s'\n", what, got.c_str(), want);
  ++failures;
}

int main() {
  {
    Device d;
    expect("one stream", d.launch(1), "o");
    expect("one stream, again", d.launch(1), "o");
    expect("a second one, the first idle", d.launch(2), "o");
    d.rt.streams[2] = StreamState::kBusy;
    expect("the first again, the second busy", d.launch(1), "1>2 c");
    expect("a third stream follows it", d.launch(3), "c");
    expect("the second again", d.launch(2), "c");
  }
  {
    Device d;
    d.launch(1);
    d.rt.streams[1] = StreamState::kBusy;
    d.rt.streams[2] = StreamState::kCapturing;
    expect("a recording beside a busy stream", d.launch(2), "c");
    expect("recorded again", d.launch(2), "c");
    expect("the first launch after a recording", d.launch(3), "3>1 c");
    expect("the next one follows it", d.launch(4), "c");
  }
  {
    Device d;
    d.launch(1);
    d.rt.streams[1] = StreamState::kCapturing;
    expect("the stream itself records", d.launch(1), "c");
    expect("it cannot be asked", d.launch(2), "c");
    d.rt.streams[1] = StreamState::kBusy;
    expect("asked as soon as it can be", d.launch(3), "3>1 c");
    expect("and once", d.launch(2), "c");
  }
  {
    Device d;
    d.launch(1);
    d.rt.streams[1] = StreamState::kBusy;
    d.rt.streams[2] = StreamState::kCapturing;
    d.launch(2);
    expect("the busy stream's own launch follows its work", d.launch(1), "c");
    expect("and all others follow that", d.launch(3), "c");
  }
  {
    Device d;
    d.launch(1);
    d.rt.streams[1] = StreamState::kGone;
    expect("a stream that is gone", d.launch(2), "wait o");
  }
  {
    Device d;
    d.launch(1);
    d.rt.streams[1] = StreamState::kBusy;
    expect("a handle per thread is put behind", d.launch(9, true), "9>1 c");
    expect("and leaves no ordinary launch after it", d.launch(1), "c");
  }
  {
    Device d;
    expect("told ahead: the first", d.ahead(1), "o");
    d.launch(1);
    d.rt.streams[2] = StreamState::kCapturing;
    expect("told ahead: one stream", d.ahead(1), "o");
    expect("told ahead: a handle per thread", d.ahead(9, true), "c");
    expect("told ahead: a recording", d.ahead(2), "c");
    expect("and none of it decides anything", d.launch(1), "o");
    d.launch(2);
    expect("told ahead: after a recording", d.ahead(1), "c");
  }
  return failures ? 1 : 0;
}
