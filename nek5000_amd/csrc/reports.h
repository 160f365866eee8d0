// Host memory that kernels report to, and the numbers of the reports (plain
// C++, no GPU code).
#pragma once

namespace nekamd {

// The thread that holds a result writes it to v and then the report's number
// to seq, where the host, waiting for that number, finds it a few microseconds
// later (a copy and a stream synchronization leave the GPU idle for about 40
// us; MI355X).
struct HostBox {
  unsigned long long seq;
  unsigned long long pad[7];
  double v[56];
};
// one report: its place and number (b null: none is made)
struct BoxRef {
  HostBox *b = nullptr;
  unsigned long long seq = 0;
};
// The reports of a solve, numbered by the count of the box's owner as they are
// handed out: a number is never given twice, also where the launch that was to
// make the report fails.  (A number given again would end the wait of a later
// solve at once, by the earlier one's report.)
struct Reports {
  HostBox *box = nullptr;  // null: none are made
  unsigned long long *count = nullptr;
  BoxRef next() const { return BoxRef{box, box ? ++*count : 0}; }
};

}  // namespace nekamd
