// The issue and wait schedule of the grouped GEMM's two LDS rings (chunk_gemm in moe_batch.hip), as plain constexpr
// C++ so that a host program can check it (tests/test_ring_schedule.py simulates the rings against it).
//
// Per wave: A (the rows) DA steps ahead in RA = DA + 1 slots, B (the wave's tiles) DB steps ahead in RB = DB + 1
// slots; OA and OB requests per step. Issue order: prologue A(0) B(0) A(1) B(1) .. A(DA-1) B(DA-1) B(DA) ..
// B(DB-1); step j then issues A(j + DA) and B(j + DB) (while < NS), after the wait for step j's data and a barrier.
// Requests complete in issue order, so waiting until at most n are outstanding completes all but the last n.
#pragma once

#include <type_traits>

namespace ijah {

// How many requests were issued after A(t) and B(t), counted at step t before it issues: the s_waitcnt vmcnt that
// makes both complete.
template <int OA, int OB, int DA, int DB>
constexpr int after_step(int t, int NS) {
  auto mn = [](int x, int y) { return x < y ? x : y; };
  auto mx = [](int x, int y) { return x > y ? x : y; };
  auto sum_ops = [&](int n) { return OA * mn(n, mx(NS - DA, 0)) + OB * mn(n, mx(NS - DB, 0)); };
  const int pa = mn(DA, NS), pb = mn(DB, NS);
  const int prologue = OA * pa + OB * pb;
  const int total = prologue + sum_ops(t);
  int last = 0;  // one past the position of the later of A(t), B(t)
  if (t < DA) {
    last = (OA + OB) * (t + 1);
  } else if (t < DB) {
    last = mx(prologue + sum_ops(t - DA) + OA, (OA + OB) * pa + OB * (t - pa) + OB);
  } else {
    last = mx(prologue + sum_ops(t - DA) + OA, prologue + sum_ops(t - DB) + ((t - DB) + DA < NS ? OA : 0) + OB);
  }
  return total - last;
}
// Steps t with t + DB < NS (both streams still issuing) wait with one compile-time count: from step DB on A(t) is the
// later request, followed by B(t - DA + DB) and DA - 1 full steps; the first DB steps have more requests behind
// theirs, so the same count waits a little longer there.
template <int DB>
constexpr bool steady_step(int t, int NS) { return t + DB < NS; }
template <int OA, int OB, int DA>
constexpr int kAfterSteady = OB + (DA - 1) * (OA + OB);
static_assert(after_step<2, 1, 2, 5>(5, 1000) == kAfterSteady<2, 1, 2> &&
                  after_step<1, 1, 2, 5>(9, 1000) == kAfterSteady<1, 1, 2> &&
                  after_step<2, 1, 1, 3>(7, 1000) == kAfterSteady<2, 1, 1>,
              "steady-state wait count");
// The count the k loop waits with at step t: the steady count, else after_step capped at 15 (the 4-bit immediate of
// wait_vm15; a larger count waits as for 15, which only waits longer).
template <int OA, int OB, int DA, int DB>
constexpr int step_wait(int t, int NS) {
  static_assert(kAfterSteady<OA, OB, DA> <= 15, "the wait's 4-bit count");
  const int n = after_step<OA, OB, DA, DB>(t, NS);
  return steady_step<DB>(t, NS) ? kAfterSteady<OA, OB, DA> : (n < 15 ? n : 15);
}

// The order itself, for the kernel and the host program alike. wait(n) makes all but the last n requests complete (n an
// integral_constant in the steady state, so that the wait takes it as an immediate), ready(s) reads what the wave itself
// requested for step s and passes the workgroup's barrier, a(j) and b(j) issue step j's requests.
template <int DA, int DB, class A, class B>
constexpr void ring_start(int NS, A a, B b) {
  for (int j = 0; j < DB && j < NS; j++) {
    if (j < DA) a(j);
    b(j);
  }
}
template <int OA, int OB, int DA, int DB, class W, class R, class A, class B>
constexpr void ring_step(int s, int NS, W wait, R ready, A a, B b) {
  if (steady_step<DB>(s, NS)) {
    wait(std::integral_constant<int, kAfterSteady<OA, OB, DA>>{});
    ready(s);
    a(s + DA);
    b(s + DB);
  } else {
    wait(step_wait<OA, OB, DA, DB>(s, NS));
    ready(s);
    if (s + DA < NS) a(s + DA);
  }
}

}  // namespace ijah
