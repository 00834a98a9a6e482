"""The host slots that the device writes block counts to (csrc/count_slots.h), without a device: which slot may be handed out
again after a call whose stream went idle, failed to answer, or answered late."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>
#include <vector>
#include "count_slots.h"
using namespace hbsa_host;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

int32_t *page() { return (int32_t *)std::calloc(kSlots * kSlotInts, sizeof(int32_t)); }

struct Scripted {   // answers of the stream, the last one for good
  std::vector<StreamState> *answers;
  StreamState operator()() const {
    const StreamState s = answers->front();
    if (answers->size() > 1) answers->erase(answers->begin());
    return s;
  }
};

int main() {
  using V = std::vector<StreamState>;
  {   // the stream's state cannot be had, or it is idle, and the ticket is not there: that slot is out of use for good
    for (StreamState end : {StreamState::kUnknown, StreamState::kIdle}) {
      CountSlots slots;
      V answers = {StreamState::kBusy, end};
      int32_t *first;
      {
        CountTicket<Scripted> t(slots, slots.take(page), Scripted{&answers});
        first = t.slot;
        t.ticket = 7;
        t.launched = true;
        CHECK(!t.wait());
      }
      first[3] = 7;   // the device writes it after all
      std::set<int32_t *> seen;
      while (int32_t *s = slots.take(page)) seen.insert(s);
      CHECK(seen.size() == kSlots - 1 && seen.count(first) == 0);
    }
  }
  {   // the same when nobody waited (an exception on the way)
    CountSlots slots;
    V answers = {StreamState::kUnknown};
    int32_t *first;
    {
      CountTicket<Scripted> t(slots, slots.take(page), Scripted{&answers});
      first = t.slot;
      t.ticket = 7;
      t.launched = true;
    }
    CHECK(slots.take(page) != first);
  }
  {   // a ticket that arrives, and a call that launched nothing, give the slot back
    CountSlots slots;
    V answers = {StreamState::kBusy};
    int32_t *first;
    {
      CountTicket<Scripted> t(slots, slots.take(page), Scripted{&answers});
      first = t.slot;
      t.ticket = 9;
      t.launched = true;
      std::thread device([&] { first[0] = 5; __atomic_store_n(first + 3, 9, __ATOMIC_RELEASE); });
      CHECK(t.wait() && t.slot[0] == 5);
      device.join();
      CHECK(slots.take(page) != first);   // (not before this call has read it)
    }
    {
      CountTicket<Scripted> t(slots, slots.take(page), Scripted{&answers});
      CHECK(t.slot == first);
    }
    CHECK(slots.take(page) == first);
  }
  {   // none left, or no page: no slot, and nothing to give back
    CountSlots slots;
    V answers = {StreamState::kBusy};
    for (int i = 0; i < kSlots; ++i) CHECK(slots.take(page) != nullptr);
    CountTicket<Scripted> t(slots, slots.take(page), Scripted{&answers});
    CHECK(t.slot == nullptr && !t.wait());
    CountSlots pageless;
    CHECK(pageless.take([] { return (int32_t *)nullptr; }) == nullptr);
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")
def test_a_slot_whose_ticket_did_not_arrive_is_not_handed_out_again(tmp_path):
    source = tmp_path / "slots.cpp"
    source.write_text(PROGRAM)
    binary = str(tmp_path / "slots")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "hbsattn_amd", "csrc"), str(source), "-o", binary],
                   check=True)
    res = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
