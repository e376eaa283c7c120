// Chip-resident time loop, FDORDER 10, viscoelastic P/SV.
#define DN_F 5
#define DN_GROUP 2
#include "dn_resident_inst.inc"
