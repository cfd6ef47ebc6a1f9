// Instantiations of the kernels over stream_tile.cuh for one (dtype, bits,
// group size) triple (the wide kernel; 8-bit: the thin grouped kernel), compiled
// once per triple with -DMQ_INST_DT=<0|1>, -DMQ_INST_BITS=<4|8> and
// -DMQ_INST_GS=<32|64|128> (a unit of all three group sizes took 4-5 minutes)
// and with -fno-slp-vectorize: the vectorizer joins the blocks' scale
// arithmetic into vectors formed after the last of them, which takes the
// dequantization out of its places between the MFMAs.
#include "dense.cuh"
#include "grouped8.cuh"

#if !defined(MQ_INST_DT) || !defined(MQ_INST_BITS) || !defined(MQ_INST_GS)
#error "compile with -DMQ_INST_DT=<0|1> -DMQ_INST_BITS=<4|8> -DMQ_INST_GS=<32|64|128>"
#endif

namespace mq {
template struct WideLaunch<MQ_INST_DT, MQ_INST_BITS, MQ_INST_GS>;
#if MQ_INST_BITS == 8
template struct Thin8Launch<MQ_INST_DT, MQ_INST_GS, false>;
template struct Thin8Launch<MQ_INST_DT, MQ_INST_GS, true>;
#endif
}  // namespace mq
