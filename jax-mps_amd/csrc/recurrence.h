// What a "recurrence" op stands for: the kernel that runs a whole loop, and how its arguments map to operands and results.
#pragma once

#include <string>

#include "codegen.h"

namespace mi355 {

// operands: the kernel's leaves, the initial states, the initial contents of stacks that are not written as a whole;
// results: the final states, then the stacks
struct RecurrenceOp {
  RecurrenceCode code;
  std::string label;            // the loop and its product, as plans name them
  size_t states = 0;
  std::vector<int> stackInit;   // per stack: operand with its initial contents, or -1 where every element is written
};

}  // namespace mi355
