// Recurrences of hybrid_recurrent.hip over prompt portions in chunks (hybrid_chunks.hip).
#pragma once
#include "hybrid_common.h"

namespace hyb {

struct MlstmChunks {
    const uint16_t *q, *k, *v;      // rows of [*, H, D] / [*, H, E], element strides per token below
    long q_row, k_row, v_row;
    const bf16_t *gi, *gf;          // raw gate pre-activations [T, H]
    long g_row;
    const float *bi, *bf;           // [H]
    float cap;
    float *state, *nstate, *mstate; // [slots,H,D,E], [slots,H,ZG,D], [slots,H,ZG], ZG = ceil(E/16)
    const int *cu_q, *positions, *slots;
    float* o;                       // [T, H, E]
    long T;                         // rows of o; those of no sequence become zeros
    int H, D, E;
    float qscale;
};

// portions (cu_q) that are long enough, up to 128 key channels, sizes in whole runs of eight and 16-byte
// addresses
bool mlstm_chunks_ok(const MlstmChunks& a, int B);
int mlstm_chunks(const MlstmChunks& a, int B, hipStream_t s);

}  // namespace hyb
