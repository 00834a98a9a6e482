// The small host-memory slots the device writes block counts to (hbsa_block_counts), one per call in flight, and the wait
// for them.  No HIP in here: the page and the stream's state come from the caller, so that both can be tested without a
// device (tests/test_count_slots.py).
#pragma once

#include <cstdint>
#include <mutex>

namespace hbsa_host {

constexpr int kSlots = 64, kSlotInts = 16;

// One page for the life of the process.  A slot is free, or with one call, or lost: a slot whose ticket was not seen to
// arrive is never handed out again, because the device may still write it, over what it writes there for a later call.
struct CountSlots {
  std::mutex m;
  int32_t *page = nullptr;
  uint64_t taken = 0;
  // nullptr when every slot is taken or there is no page (`make_page`: kSlots * kSlotInts zeros the device can write, or nullptr)
  template <typename MakePage>
  int32_t *take(MakePage &&make_page) {
    std::lock_guard<std::mutex> lock(m);
    if (page == nullptr) page = make_page();
    if (page == nullptr || taken == ~0ull) return nullptr;
    const int i = __builtin_ctzll(~taken);
    taken |= 1ull << i;
    return page + i * kSlotInts;
  }
  void give_back(int32_t *slot) {
    std::lock_guard<std::mutex> lock(m);
    taken &= ~(1ull << ((slot - page) / kSlotInts));
  }
};

enum class StreamState { kBusy, kIdle, kUnknown };   // kUnknown: the question itself failed

// Waits until the device has written `ticket` behind the counts.  Looks at memory instead of waiting for an event: the
// answer arrives while later launches of the same stream are already running.  False: the stream is idle, or its state
// cannot be had, and the ticket is not there (a stream of unknown state may still write it).
template <typename State>
bool wait_for_ticket(const int32_t *slot, int32_t ticket, State &&stream_state) {
  const auto arrived = [&]() { return __atomic_load_n(slot + 3, __ATOMIC_ACQUIRE) == ticket; };
  for (unsigned spins = 1;; ++spins) {
    if (arrived()) return true;
    __builtin_ia32_pause();
    if ((spins & 0xfffu) == 0 && stream_state() != StreamState::kBusy) return arrived();
  }
}

// A slot for the time of one call.  wait() ends the launch that writes it; without one the destructor waits.
template <typename State>
struct CountTicket {
  CountSlots &slots;
  State state;
  int32_t *slot;
  int32_t ticket = 0;
  bool launched = false;   // from the launch on (also one that reported an error: it may be an earlier one's)
  CountTicket(CountSlots &slots_, int32_t *slot_, State state_) : slots(slots_), state(state_), slot(slot_) {}
  CountTicket(const CountTicket &) = delete;
  CountTicket &operator=(const CountTicket &) = delete;
  // True: the counts have arrived and stay valid until this object goes.
  bool wait() {
    if (slot == nullptr || !launched) return false;
    if (!wait_for_ticket(slot, ticket, state)) {
      slot = nullptr;   // lost
      return false;
    }
    launched = false;
    return true;
  }
  ~CountTicket() {
    if (launched) (void)wait();
    if (slot != nullptr) slots.give_back(slot);
  }
};

}  // namespace hbsa_host
