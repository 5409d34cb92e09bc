// Internal declarations shared by the library's translation units.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/krafla_hip.h"

hipStream_t kr_stream(void);
// records the first error (sticky) with a message
void kr_fail(ml_status st, const char *what, hipError_t e);
// records a launch error, if any
void kr_check_launch(const char *what);

// devices whose static scratch addresses the library keeps
constexpr int KR_MAX_DEVICES = 16;
// kr_attn.hip: takes this device's address of the attention scratch array
ml_status kr_attn_setup(int dev);
// kr_family.hip: soft-caps the attention scratch's scores in place, in the
// layout the attention launches of ntok tokens use
void kr_softcap_scores(float *att, int n_heads, int max_seq, int window, const int *pos, int ntok, float cap);
// kr_matvec_short.hip: launches a normalizing matvec whose sum is short; args
// is the caller's MvArgs (kr_matvec.h)
void kr_matvec_short(int epi, bool mixed, int type, int d16, const void *args, size_t bytes, int grid, size_t lds);
