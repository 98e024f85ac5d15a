// The library with MKV_PLAN_TABLE_GROUPS 0 (the plan pass's record workgroups make the
// rotation tables), so that the tests run that build of the plan pass too.
#define MKV_PLAN_TABLE_GROUPS 0
#include "kvshift.hip"
