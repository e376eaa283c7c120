// Chip-resident time loop, FDORDER 10, isotropic P/SV.
#define DN_F 5
#define DN_GROUP 0
#include "dn_resident_inst.inc"
