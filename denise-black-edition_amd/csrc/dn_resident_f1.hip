// Chip-resident time loop, FDORDER 2, isotropic P/SV.
#define DN_F 1
#define DN_GROUP 0
#include "dn_resident_inst.inc"
