// span.hpp -- substeps that are planned on the host a few at a time, ahead of
// their launches.
//
// Planning a substep moves the host's bookkeeping on (time, sort counters,
// which particle copy is current), so that the next one can be planned. An
// error must not leave it ahead of the device: a planning error still runs the
// substeps planned before it, a launch error stops there, and either way the
// bookkeeping goes back to the start of the first substep that did not run.
#pragma once

#include <cstdint>
#include <vector>

namespace mpm_engine {

// At least one substep (n >= 1) and at most n. `ops` has
//   State save()          the bookkeeping as it is
//   void restore(State)   back to it
//   int plan(i)           plans substep i and moves the bookkeeping on
//   bool more(planned)    whether a further one belongs to the span
//   int begin()           once all are planned, ahead of the launches
//   int launch(i)
//   int end()             after the launches, whatever they returned
// which return 0 or an error. *ran: the substeps launched. Returns the first
// error.
template <class Ops>
int run_span(Ops& ops, int32_t n, int32_t* ran) {
  std::vector<decltype(ops.save())> before;
  *ran = 0;
  int error = 0;
  int32_t planned = 0;
  do {
    before.push_back(ops.save());
    error = ops.plan(planned);
    if (error) {
      ops.restore(before.back());
      break;
    }
    ++planned;
  } while (planned < n && ops.more(planned));
  int rc = planned > 0 ? ops.begin() : 0;
  while (!rc && *ran < planned) {
    rc = ops.launch(*ran);
    if (!rc) ++*ran;
  }
  if (*ran < planned) ops.restore(before[(size_t)*ran]);
  const int re = ops.end();
  if (rc) return rc;
  return error ? error : re;
}

}  // namespace mpm_engine
