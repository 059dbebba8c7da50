// The complex64 instantiations of g4_tiled.hip.
#define G4_TILED_FLOAT
#include "g4_tiled.hip"
