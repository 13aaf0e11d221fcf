// The cut of a staged copy, for tests/test_copy_plan.py (built there with g++).
#include "../nimblesm_amd/csrc/nsm_copy_plan.h"

extern "C" void copy_plan(size_t bytes, size_t out[4])
{
  const nsm::CopyPlan p = nsm::copy_plan(bytes);
  out[0]                = p.chunk;
  out[1]                = (size_t)p.own;
  out[2]                = (size_t)p.helpers;
  out[3]                = p.pinned();
}
