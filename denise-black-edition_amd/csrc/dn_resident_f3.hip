// Chip-resident time loop, FDORDER 6, isotropic P/SV.
#define DN_F 3
#define DN_GROUP 0
#include "dn_resident_inst.inc"
