/* The convergence flag's rules (wildfires_amd/csrc/hip/wf_iter.h) for the CPU
 * check in tests/test_pressure_passes.py; test code only. */
#include "../../wildfires_amd/csrc/hip/wf_iter.h"

int iter_flag(int ended, int m) { return wf_iter_flag(ended, m); }
int first_pass_returns(int flag, int check) { return wf_first_pass_returns(flag, check); }
int pass_returns(int flag) { return wf_pass_returns(flag); }
