// Chip-resident time loop, FDORDER 8, isotropic P/SV.
#define DN_F 4
#define DN_GROUP 0
#include "dn_resident_inst.inc"
