// The state behind fl_state_create: shared by the decode / verify launches and the prompt pass.
#pragma once
#include "fl_common.h"

struct fl_state {
  fl_model_desc d;
  int max_seq;
  int grid;   // decode workgroups (1 per CU)
  int vgrid;  // verify workgroups (1 per CU)
  uint16_t *kc, *vc;
  uint32_t *h, *attn, *act;
  unsigned long long* qkv;
  unsigned long long* part;
  uint16_t* vrows;              // verify exchange rows: h [FL_MAX_VERIFY][D], attn [..][D], act [..][F]
  unsigned long long* vpart;    // verify attention slice partials [NH][VNS][FL_MAX_VERIFY][66]
  uint32_t* vflag;              // verify ready flags
  uint32_t* shist;              // fused sampling exchange: per-workgroup histograms
  unsigned long long* sword;    // ... bin totals, maxima, partial sums
  int att_spw, gq_min, gq_kps;
  int defer_min;  // key slices from which the per-head attention leaves its merge to the O phase
  int vkps, vtok_work;
  int coop;       // launch with hipLaunchCooperativeKernel (else a plain launch, the default)
  // the k_decode instantiations of the chunk budget that fits the model, by attention: per-head
  // units (0), with the slice merge deferred to the O phase (1), by KV group (2; small budget only,
  // else null)
  const void* kdec[3];
  int verify_ok;  // k_verify's dynamic LDS fits and a grid of it is co-resident
  unsigned long long* amax;
  uint32_t* done;
  int32_t* err;
  uint32_t epoch;
  unsigned long long* prof;
  int prof_slots;
  unsigned long long spin_ticks;  // wait bound passed to every launch
  uint32_t* stall;                // zero word, never written: forced-timeout wait (tests)
  int force_timeout;
  void* blocks[16];
  int nblocks;
  void* uc[12];  // pooled uncached exchange buffers
  size_t uc_bytes[12];
  int nuc;
  // Tags are 16 bits (1..65535) and advance 5 per layer per launch, so a word left over from an
  // older launch could carry the tag a reader is waiting for once the tags have gone round. The
  // exchange buffers are zeroed (tag 0: never valid) every clear_period launches, fewer than
  // take the tags round.
  uint32_t clear_period, since_clear;
};

// every pointer that all entry points need is set (fl_decode.hip)
bool fl_weights_ok(const fl_weights* w);
