"""The grouped GEMM's ring schedule (ijah_amd/csrc/ring_schedule.h, used by chunk_gemm in moe_batch.hip), compiled
for the host and checked against an event simulation of the two rings: at every step the wait count the kernel uses
must leave both of that step's operands complete, and no ring slot may be refilled before its previous step consumed
it. Requests complete in issue order (the hardware's vector-memory counter rule the waits rely on).

The simulation shares no code with the header: it replays the issue order chunk_gemm follows (prologue A(0) B(0) ..
A(DA-1) B(DA-1) B(DA) .. B(DB-1); step s issues A(s + DA) and B(s + DB) after its wait and barrier) and records
where each request sits."""
import subprocess

import pytest

from conftest import ROOT

# (OA, OB, DA, DB): requests per A / B step and lead, for the shapes chunk_gemm instantiates (32- and 128-row chunks:
# DA 2, DB 5 at K < 6 and DA 1, DB 3 at K >= 6; 64-row chunks: DA 1, DB 3 at every K; OA 2 for the two-operand 128-row A,
# else 1; every B step is one request)
CONFIGS = [(2, 1, 2, 5), (1, 1, 2, 5), (2, 1, 1, 3), (1, 1, 1, 3)]
MAX_NS = 80


@pytest.fixture(scope="module")
def waits(tmp_path_factory):
    d = tmp_path_factory.mktemp("ring")
    src = d / "ring.cpp"
    lines = ['#include <cstdio>', '#include "ring_schedule.h"', "int main() {"]
    for oa, ob, da, db in CONFIGS:
        lines.append(f"  for (int ns = 1; ns <= {MAX_NS}; ns++) for (int t = 0; t < ns; t++) "
                     f'std::printf("{oa} {ob} {da} {db} %d %d %d\\n", ns, t, ijah::step_wait<{oa}, {ob}, {da}, {db}>(t, ns));')
    lines.append("  return 0;\n}")
    src.write_text("\n".join(lines))
    exe = d / "ring"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'ijah_amd' / 'csrc'}", str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    w = {}
    for line in out.splitlines():
        oa, ob, da, db, ns, t, n = map(int, line.split())
        w[(oa, ob, da, db, ns, t)] = n
    return w


def simulate(oa, ob, da, db, ns, wait):
    """Replays the issue order; returns the list of problems found (empty when the schedule is sound)."""
    issued = []  # request tags in issue order: ("A", step) or ("B", step), OA or OB entries per step
    slot_a, slot_b = {}, {}  # ring slot -> the step whose data it holds
    problems = []

    def issue(kind, j, now):
        ring, nslots = (slot_a, da + 1) if kind == "A" else (slot_b, db + 1)
        sl = j % nslots
        prev = ring.get(sl)
        if prev is not None and prev >= now:  # the previous occupant is consumed at its own step, before `now`
            problems.append(f"{kind}({j}) overwrites {kind}({prev}) in slot {sl} at step {now}")
        ring[sl] = j
        issued.extend([(kind, j)] * (oa if kind == "A" else ob))

    for j in range(min(db, ns)):  # prologue
        if j < da:
            issue("A", j, 0)
        issue("B", j, 0)
    for t in range(ns):
        done = len(issued) - wait(t)  # requests complete in issue order
        for kind in ("A", "B"):
            last = max(i for i, r in enumerate(issued) if r == (kind, t))
            if last >= done:
                problems.append(f"NS={ns} step {t}: {kind}({t}) may be outstanding after the wait")
        ring, nslots = (slot_a, da + 1), (slot_b, db + 1)
        if slot_a.get(t % (da + 1)) != t or slot_b.get(t % (db + 1)) != t:
            problems.append(f"NS={ns} step {t}: a ring slot does not hold step {t}")
        if t + da < ns:
            issue("A", t + da, t)
        if t + db < ns:
            issue("B", t + db, t)
    return problems


@pytest.mark.parametrize("cfg", CONFIGS, ids=lambda c: "OA{}_OB{}_DA{}_DB{}".format(*c))
def test_ring_schedule_waits_and_slots(waits, cfg):
    oa, ob, da, db = cfg
    for ns in range(1, MAX_NS + 1):
        probs = simulate(oa, ob, da, db, ns, lambda t: waits[(oa, ob, da, db, ns, t)])
        assert not probs, probs[:5]


def test_ring_schedule_waits_are_not_wasteful(waits):
    """In the steady state the wait leaves exactly the later step requests outstanding: a wait count one larger
    would let the step's own data be outstanding (so the count is the tightest sound one)."""
    oa, ob, da, db = CONFIGS[0]
    ns = MAX_NS
    probs = simulate(oa, ob, da, db, ns, lambda t: waits[(oa, ob, da, db, ns, t)] + 1)
    assert probs, "a looser wait was not caught: the simulation would not see a too-late wait"


@pytest.fixture(scope="module")
def events(tmp_path_factory):
    """The waits, reads and requests of the k loop itself: ring_start and ring_step, the templates that chunk_gemm
    expands, run on the host with callbacks that print."""
    d = tmp_path_factory.mktemp("ring_loop")
    src, exe = d / "loop.cpp", d / "loop"
    lines = ['#include <cstdio>', '#include "ring_schedule.h"', "int main() {",
             '  auto a = [](int j) { std::printf(" A%d", j); };', '  auto b = [](int j) { std::printf(" B%d", j); };',
             '  auto w = [](auto n) { std::printf(" w%d", (int)n); };',
             '  auto r = [](int s) { std::printf(" r%d", s); };']
    for oa, ob, da, db in CONFIGS:
        lines += [f"  for (int ns = 1; ns <= {MAX_NS}; ns++) {{", f'    std::printf("{oa} {ob} {da} {db} %d", ns);',
                  f"    ijah::ring_start<{da}, {db}>(ns, a, b);",
                  f"    for (int s = 0; s < ns; s++) ijah::ring_step<{oa}, {ob}, {da}, {db}>(s, ns, w, r, a, b);",
                  '    std::printf("\\n");', "  }"]
    src.write_text("\n".join([*lines, "  return 0;", "}"]))
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'ijah_amd' / 'csrc'}", str(src), "-o", str(exe)], check=True)
    got = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        f = line.split()
        got[tuple(map(int, f[:5]))] = [(e[0], int(e[1:])) for e in f[5:]]
    return got


@pytest.mark.parametrize("cfg", CONFIGS, ids=lambda c: "OA{}_OB{}_DA{}_DB{}".format(*c))
def test_ring_loop_runs_the_checked_schedule(waits, events, cfg):
    """The kernel's own loop issues in the order that the simulation replays, waits with the counts that it checks, and
    reads each step once, in order, between the wait and the requests that reuse its predecessor's slots. Every count
    fits the wait's 4-bit field."""
    oa, ob, da, db = cfg
    for ns in range(1, MAX_NS + 1):
        want = []
        for j in range(min(db, ns)):
            want += ([("A", j)] if j < da else []) + [("B", j)]
        for t in range(ns):
            want += [("w", waits[(*cfg, ns, t)]), ("r", t)]
            want += [("A", t + da)] if t + da < ns else []
            want += [("B", t + db)] if t + db < ns else []
        assert events[(*cfg, ns)] == want, ns
        assert all(0 <= n <= 15 for k, n in want if k == "w")


def test_grouped_gemm_expands_the_checked_loop():
    """chunk_gemm has no wait or request order of its own beside the templates above."""
    src = (ROOT / "ijah_amd" / "csrc" / "moe_batch.hip").read_text()
    body = src[src.index("void chunk_gemm("):src.index("Hadamard on")]
    assert body.count("ring_start<") == 1 and body.count("ring_step<") == 1
    # one wait of each form, inside the callbacks; the requests of the prologue and of the step
    assert body.count("s_waitcnt(") == 1 and body.count("wait_vm15(") == 1
    assert body.count("issue_a(") == 2 and body.count("issue_b(") == 2
