// Chip-resident time loop, FDORDER 12, isotropic P/SV.
#define DN_F 6
#define DN_GROUP 0
#include "dn_resident_inst.inc"
