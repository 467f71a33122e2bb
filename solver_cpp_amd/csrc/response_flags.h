// Whether a context's pivoting list and terminally-ill flag are clear on its
// stream (host only, no HIP).
#pragma once

namespace sca {

// A material-point update appends to the pivoting list and raises the flag, so
// both are cleared before it.  An evaluation whose last kernels clear them for
// the next one saves that launch; only its return says that those kernels are
// on the stream.  An evaluation that throws may have left entries behind (the
// list has room for one update's), so from its start until its return they
// count as not clear.
class ResponseFlags {
 public:
  // launch(clear): one evaluation's launches, clearing the list and the flag
  // first when clear is true; cleared: they end with both clear
  template <typename Launch>
  void evaluation(bool cleared, Launch&& launch) {
    const bool clear = !clean_;
    clean_ = false;
    launch(clear);
    clean_ = cleared;
  }
  // they are written outside an evaluation
  void written() { clean_ = false; }

 private:
  bool clean_ = false;
};

}  // namespace sca
