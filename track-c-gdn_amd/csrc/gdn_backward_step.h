// The training step's backward, called by the package's autograd operator.
#pragma once

#include <stddef.h>
#include <stdint.h>

// gdn_prefill_bwd (include/gdn_hip.h) carried through the gating in the same
// launches: every token gradient in bf16, the inputs' own type (dq, dk
// [T, HQ, 128], dv [T, HV, 128], da, db [T, HV]), and dA_log, ddt_bias [HV]
// fp32, written whole (zeros when the batch holds no token).  Equal to
// gdn_prefill_bwd, gdn_gate_bwd and a rounding of the token gradients, up to
// the order of the two per-head sums.  Same workspace and status codes.
extern "C" int gdn_prefill_bwd_step(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                    const float* A_log, const uint16_t* a, const float* dt_bias,
                                    const uint16_t* b, const void* cu_seqlens, int cu_is_int32, int N,
                                    int T, int HQ, int HV, float scale, const uint16_t* h, int h_chunks,
                                    const uint16_t* d_out, const float* d_final_state, uint16_t* dq,
                                    uint16_t* dk, uint16_t* dv, uint16_t* da, uint16_t* db, float* dA_log,
                                    float* ddt_bias, float* d_initial_state, void* workspace,
                                    size_t workspace_bytes, void* stream);
