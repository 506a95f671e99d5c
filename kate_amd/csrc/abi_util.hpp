// abi_util.hpp -- helpers shared by the C-ABI translation units.
#pragma once

#include <string>

#include "kate_hip.h"
#include "plan.hpp"

namespace kate {
int set_error(int code, const std::string& msg);
std::string program_from_abi(const kate_program* in, Program& p);
std::string plan_options(const kate_options& opt, PlanOptions& po);
// Whether every shape and form is left to the planner, so that it may use
// streamed passes (PlanOptions::stream).
bool may_stream(const kate_options& opt, const PlanOptions& po);
// Whether dense gates of 4 to 6 qubits may run on the matrix cores
// (PlanOptions::gate_mfma).
bool may_gate_mfma(const kate_options& opt, const PlanOptions& po);
// The tile of a program of fewer than 12 qubits whose shapes are left to
// the planner.
void fit_tile(int tile_qubits, int low_qubits, int nqubits, PlanOptions& po);
}  // namespace kate
