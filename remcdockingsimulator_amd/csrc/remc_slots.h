// remc_slots.h -- when the members of a replica may reuse a bank of slots.
//
// The workgroups (members) of a replica add their partial sums through two banks
// of tagged slots in device memory.  Every member counts the exchanges it has
// been through; the count's parity selects the bank.  A member writes the bank
// of exchange n again in exchange n + 2, after it has seen every member's
// partial of exchange n + 1, which each wrote after it had read all of exchange
// n: that exchange n + 1 took place is what orders the two uses.  So the count
// advances only with an exchange.  (Counting a window that publishes nothing put
// the next exchange into the bank of the last one, where a member still polling
// could find its tag overwritten, spin to its limit and fail the launch.)
#pragma once

#include "remc_math.h"

// The count after a window of `slots` slots, of which `still` leave their bead
// where it is: those have no partial, and a window of nothing else no exchange.
// Both numbers are the same in every member.
REMC_HD unsigned int remc_exchanges_after_window(unsigned int n, int slots, int still)
{
    return still < slots ? n + 1u : n;
}
