// Chip-resident time loop, FDORDER 4, isotropic P/SV.
#define DN_F 2
#define DN_GROUP 0
#include "dn_resident_inst.inc"
